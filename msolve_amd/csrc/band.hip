// Band Cholesky factorization and triangular sweeps (direct solver, first-
// sample preconditioner, coarsest multigrid levels): SkylineMatrix2D.
// Factorize / Solve (SkylineMatrix2D.cs:63-212) in blocks of kBandNB = 64
// columns.  Lower band storage band[j*bW + (i - j)], bW >= bandwidth + 64,
// so every panel is a full rectangle (entries outside the true band stay
// zero).  grid.y = sample of the class.
//
// A factorization runs k_chol_block, k_chol_panel_inv and k_chol_update_mfma
// per block (zero-energy modes: k_chol_diag and k_chol_panel in their place,
// and k_band_linv at the end).
//
// A sweep walks the factor in blocks of kBandNB = 64 columns, and a block
// depends on the one before: the time is the number of blocks times the
// latency of one.  So the 64 x 64 diagonal blocks are inverted once per
// factorization (in k_chol_block, whose panel needs the inverse too; with
// zero-energy modes by k_band_linv, all blocks at once), which turns each
// serial 64-step substitution into a 64 x 64 product of one parallel step.
// The inverse takes the block's place in the band, so a factor is n W doubles
// and nothing beside it.  Both sweeps push a solved block's contribution
// outwards (forward: the rows below; backward: the rows above), so no block
// waits on a reduction over rows that another workgroup holds.
//
// Measured, factorization (MI355X, one 16^3 sample, 217 blocks of width 960):
// 218 -> 41 us per block, 47 -> 8.9 ms: the diagonal block 137 -> 26 us (the
// chain of 64 pivots; it was a 64-step loop with two barriers a step), the
// panel 58 -> 5 us (a product with the inverse instead of a column sweep),
// the update 23 -> 10.6 us (matrix cores instead of 4 x 4 register tiles
// through LDS).
//
// Measured, sweeps: against a launch pair per block and sweep with 64-step
// substitutions, eight first-sample solves of 12^3 (6084 rows, width 576, 22
// applications) 525 -> 37.5 ms, the sweeps of a 16^3 direct solve (13872 rows)
// 48 -> 1.6 ms.  Wide bands take a launch per block, narrow ones both sweeps
// in one launch and one workgroup, whose CU then loads the whole panel (width
// 512: 62 GB/s).  us a block and sweep, with an iteration's other kernels:
//   samples, width     1, 576   8, 320   8, 512   8, 576   64, 320   64, 512   64, 576
//   launch per block     12.3     3.66     3.71     3.59      3.78      4.57      4.63
//   one launch            4.8     4.06     4.26     4.51      4.06      4.22      4.42
// (one sample: the first application, which is not captured).  The line lies
// at width 512: up to there a launch per block gains at most 15%, and loses 8%
// with many samples, while in one launch an idle multigrid cycle costs next to
// nothing (17 ragged samples, width 384: 85 against 203 ms, when cycles still
// ran idle) and uncaptured launches a third; wider, few samples lose 25% in
// one launch, and eight waves of 64 rows end it at 576 anyway.
#include <hip/hip_runtime.h>

#include "msa_common.hpp"

namespace msa {

namespace {

constexpr int kSweepWaves = 8;

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
// two neighbouring factor entries at any 8-byte boundary
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

// Pointers kept in ClassDev are generic: global_* loads instead of flat_*.
template <typename X>
__device__ __forceinline__ __attribute__((address_space(1))) X *glob(X *p)
{
    return (__attribute__((address_space(1))) X *)p;
}
#define GLOB __attribute__((address_space(1)))

// v of lane `CTRL(lane)` within 16 lanes, as two 32-bit DPP moves.
template <int CTRL>
__device__ __forceinline__ double dpp16(double v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// Sum over each aligned group of 8 lanes, in every lane of the group:
// quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror.
__device__ __forceinline__ double sum8(double v)
{
    v += dpp16<0xB1>(v);
    v += dpp16<0x4E>(v);
    v += dpp16<0x141>(v);
    return v;
}

// ---------------------------------------------------- diagonal block inverse

// Register v of lane l in v_mfma_f64_16x16x4: the operands are A[l % 16][l / 16]
// and B[l / 16][l % 16], the result D[l / 16 + 4 v][l % 16].  So a product's
// registers v = 0..3 are the B operands of the next one's four steps.
#define MFMA64(a, b, c) __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0)

typedef double Tile64[kBandNB][kBandNB + 1];  // in LDS, a column apart per row

// X = L^-1 of a 64 x 64 lower triangle in LDS by 256 threads, rd = 1 / diag:
// the four 16 x 16 diagonal blocks by substitution (wave w, lane = column),
// then the blocks below by distance d from the diagonal,
// X_ij = -X_ii sum_k L_ik X_kj, one block per wave on the matrix cores.
__device__ __forceinline__ void invert_lower(const Tile64 &L, Tile64 &X, const double *rd, int t)
{
    const int lane = t & 63, w = t >> 6, o = 16 * w;
    for (int e = t; e < kBandNB * kBandNB; e += 256) X[e >> 6][e & 63] = 0.0;
    __syncthreads();
    if (lane < 16) {
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = i == lane ? 1.0 : 0.0;
#pragma unroll
        for (int k = 0; k < 16; k++) {
            x[k] *= rd[o + k];
#pragma unroll
            for (int i = k + 1; i < 16; i++) x[i] -= L[o + i][o + k] * x[k];
        }
#pragma unroll
        for (int i = 0; i < 16; i++) X[o + i][o + lane] = x[i];
    }
    const int r = lane & 15, g = lane >> 4;
    for (int d = 1; d < 4; d++) {
        __syncthreads();
        const int i = d + w, j = w;
        if (i < 4) {
            f64x4 s = {0, 0, 0, 0};
            for (int k = j; k < i; k++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    s = MFMA64(L[16 * i + r][16 * k + 4 * q + g], X[16 * k + 4 * q + g][16 * j + r], s);
            f64x4 p = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 4; q++) p = MFMA64(X[16 * i + r][16 * i + 4 * q + g], s[q], p);
#pragma unroll
            for (int v = 0; v < 4; v++) X[16 * i + g + 4 * v][16 * j + r] = -p[v];
        }
    }
    __syncthreads();
}

// The inverse takes the block's place in the band: it is a lower triangle too,
// and nothing reads the block itself once its panel is formed.
__device__ __forceinline__ void store_inverse(const ClassDev &C, GLOB double *AB, int k0, const Tile64 &X,
                                              int t)
{
    const int nk = min(kBandNB, C.bn - k0);
    for (int e = t; e < kBandNB * kBandNB; e += 256) {
        const int c = e >> 6, r = e & 63;
        if (r >= c && r < nk) AB[(size_t)(k0 + c) * C.bW + (r - c)] = X[r][c];
    }
}

// Lower triangle of the diagonal block at column k0 into LDS, zeros above;
// rows past the band's end (a last, partial block) become identity rows.
__device__ __forceinline__ void load_diag(const ClassDev &C, const GLOB double *AB, int k0, Tile64 &L,
                                          int t)
{
    const int nk = min(kBandNB, C.bn - k0);
    for (int e = t; e < kBandNB * kBandNB; e += 256) {
        const int c = e >> 6, r = e & 63;
        L[r][c] = r >= c && r < nk ? AB[(size_t)(k0 + c) * C.bW + (r - c)] : (r == c ? 1.0 : 0.0);
    }
}

// Inverse of every diagonal block of every factor, in place: grid (block,
// sample).
__global__ __launch_bounds__(256) void k_band_linv(const ClassDev *__restrict__ cp)
{
    __shared__ Tile64 L, X;
    __shared__ double rd[kBandNB];
    const ClassDev &C = *cp;
    const int t = threadIdx.x, smp = blockIdx.y;
    const int k0 = blockIdx.x * kBandNB;
    GLOB double *AB = glob(C.band + (size_t)smp * C.band_ss);
    load_diag(C, AB, k0, L, t);
    __syncthreads();
    if (t < kBandNB) rd[t] = 1.0 / L[t][t];
    __syncthreads();
    invert_lower(L, X, rd, t);
    store_inverse(C, AB, k0, X, t);
}

// ------------------------------------------------------------ factorization

__device__ __forceinline__ double lane_f64(double v, int l)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, l);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), l);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Cholesky of the diagonal block at column k0 and its inverse, one workgroup
// per sample: columns in four groups of 16, each factored by wave 0 with
// lane = row and the group in registers (a pivot's reciprocal root from
// v_rsq_f64 and one cubic Newton step), then applied to the columns right of
// it on the matrix cores.  The chain of 64 pivots is what takes the time.
__global__ __launch_bounds__(256) void k_chol_block(const ClassDev *__restrict__ cp, int k0)
{
    __shared__ Tile64 L, X;
    __shared__ double rd[kBandNB];
    const ClassDev &C = *cp;
    const int smp = blockIdx.y, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    GLOB double *AB = glob(C.band + (size_t)smp * C.band_ss);
    load_diag(C, AB, k0, L, t);
    __syncthreads();
    bool fail = false;
    const int r = lane & 15, g = lane >> 4;
    for (int b = 0; b < 4; b++) {
        const int o = 16 * b;
        if (wave == 0) {
            double a[16];
#pragma unroll
            for (int c = 0; c < 16; c++) a[c] = L[lane][o + c];
#pragma unroll
            for (int c = 0; c < 16; c++) {
                double d = lane_f64(a[c], o + c);
                if (!(d > 0.0) || !isfinite(d)) {
                    fail = true;
                    d = 1.0;
                }
                double y = __builtin_amdgcn_rsq(d);
                const double e = __builtin_fma(-(d * y), y, 1.0);
                y = __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
                const double l = lane > o + c ? a[c] * y : 0.0;
#pragma unroll
                for (int c2 = c + 1; c2 < 16; c2++) a[c2] -= l * lane_f64(l, o + c2);
                double s = d * y;
                s = __builtin_fma(0.5 * y, __builtin_fma(-s, s, d), s);
                a[c] = lane == o + c ? s : l;
                if (lane == 0) rd[o + c] = y;
            }
#pragma unroll
            for (int c = 0; c < 16; c++) L[lane][o + c] = a[c];
        }
        __syncthreads();
        // columns right of the group: tiles (I, J), b < J <= I
        for (int T = wave, I = b + 1, J = b + 1; I < 4; ) {
            if (T == 0) {
                f64x4 s = {0, 0, 0, 0};
#pragma unroll
                for (int q = 0; q < 4; q++)
                    s = MFMA64(L[16 * I + r][o + 4 * q + g], L[16 * J + r][o + 4 * q + g], s);
#pragma unroll
                for (int v = 0; v < 4; v++) L[16 * I + g + 4 * v][16 * J + r] -= s[v];
                T = 4;
            }
            T--;
            if (++J > I) {
                I++;
                J = b + 1;
            }
        }
        __syncthreads();
    }
    if (t == 0 && fail) C.bfail[smp] = 1;
    invert_lower(L, X, rd, t);
    store_inverse(C, AB, k0, X, t);
}

// Panel rows [r0, r0 + m), r0 = k0 + 64: L21 = A21 L11^-T as a product with
// the inverted block, 16 rows per wave, straight from and to global memory:
// D[c][row] = sum_k Linv[c][k] A21[row][k], so that loads and stores run
// along rows.  (Rows past the band's end hold zeros.)
__global__ __launch_bounds__(256) void k_chol_panel_inv(const ClassDev *__restrict__ cp, int k0, int m)
{
    const ClassDev &C = *cp;
    const int smp = blockIdx.y, lane = threadIdx.x & 63;
    const int r = lane & 15, g = lane >> 4, W = C.bW;
    const int i0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16;  // row - r0
    if (i0 >= m) return;
    GLOB double *P = glob(C.band + (size_t)smp * C.band_ss) + (size_t)k0 * W + kBandNB + i0 + r;
    // entry (row, col) of the inverse (col <= row) at LI[col (W - 1) + row]
    const GLOB double *LI = glob((const double *)C.band + (size_t)smp * C.band_ss) + (size_t)k0 * W;
    double a[16];  // A21[row][4 q + g]
#pragma unroll
    for (int q = 0; q < 16; q++) a[q] = P[(size_t)(4 * q + g) * (W - 1)];
    f64x4 s[4];
#pragma unroll
    for (int ct = 0; ct < 4; ct++) {
        s[ct] = f64x4{0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < 4 * (ct + 1); q++) {
            const double l = LI[(size_t)(4 * q + g) * (W - 1) + 16 * ct + r];
            const bool low = q < 4 * ct || r >= 4 * (q - 4 * ct) + g;
            s[ct] = MFMA64(low ? l : 0.0, a[q], s[ct]);
        }
    }
    if (i0 + r >= m) return;
#pragma unroll
    for (int ct = 0; ct < 4; ct++)
#pragma unroll
        for (int v = 0; v < 4; v++) P[(size_t)(16 * ct + g + 4 * v) * (W - 1)] = s[ct][v];
}

// Trailing update of the band window: A[i][j] -= sum_c L[i][k0+c] L[j][k0+c]
// for r0 <= j <= i < r0 + m; one workgroup per 64 x 64 tile (I, J), J <= I,
// a 32 x 32 part per wave: D[j][i], operands straight from the panel (each
// load four 128-byte row pieces).
__global__ __launch_bounds__(256) void k_chol_update_mfma(const ClassDev *__restrict__ cp, int k0, int m)
{
    const ClassDev &C = *cp;
    const int smp = blockIdx.y, W = C.bW;
    // tile index -> (I, J) with J <= I
    const int tix = blockIdx.x;
    int I = (int)((sqrt(8.0 * tix + 1.0) - 1.0) * 0.5);
    while ((I + 1) * (I + 2) / 2 <= tix) I++;
    while (I * (I + 1) / 2 > tix) I--;
    const int J = tix - I * (I + 1) / 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, g = lane >> 4;
    const int i0 = I * kBandNB + 32 * (wave & 1), j0 = J * kBandNB + 32 * (wave >> 1);
    if (i0 + 31 < j0 || i0 >= m || j0 >= m) return;
    GLOB double *AB = glob(C.band + (size_t)smp * C.band_ss);
    const GLOB double *P = AB + (size_t)k0 * W + kBandNB + (size_t)g * (W - 1) + r;
    f64x4 s[2][2];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int v = 0; v < 2; v++) s[u][v] = f64x4{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const GLOB double *Pq = P + (size_t)(4 * q) * (W - 1);
        const double a0 = Pq[j0], a1 = Pq[j0 + 16], b0 = Pq[i0], b1 = Pq[i0 + 16];
        s[0][0] = MFMA64(a0, b0, s[0][0]);
        s[0][1] = MFMA64(a0, b1, s[0][1]);
        s[1][0] = MFMA64(a1, b0, s[1][0]);
        s[1][1] = MFMA64(a1, b1, s[1][1]);
    }
    const int r0 = k0 + kBandNB;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
        for (int w = 0; w < 2; w++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int j = j0 + 16 * u + g + 4 * v, i = i0 + 16 * w + r;
                if (i >= j && i < m) AB[(size_t)(r0 + j) * W + (i - j)] -= s[u][w][v];
            }
}

// ------------------------------------------------------------------- sweeps

// Range-checked view of `bytes` bytes at p (the same in the whole wave):
// loads past the end return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wave_view(const GLOB double *p, unsigned bytes)
{
    const unsigned long long a = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void *)(((unsigned long long)hi << 32) | lo), (short)0,
                                             (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// Row t / 8 of the inverted block (backward: of its transpose) times the
// block's right-hand side y: lane p of the 8 of a row takes columns 2 p + 16 j
// (+ 1), so that a backward load covers 128 contiguous bytes, and the 8 lanes
// sum by DPP.  The block lies in the band at byte `base` of the view `ab`,
// entry (row, col) at col (W - 1) + row; `out` is an offset past the view.
// Backward, the entries of the other triangle are the unused (zero) end of
// the column before; columns past the band's end (a last, partial block) are
// out of range.
struct LinvRow {
    f64x2 v[4];
};
template <bool FWD>
__device__ __forceinline__ LinvRow load_linv(__amdgpu_buffer_rsrc_t ab, unsigned base, unsigned out, int W,
                                             int t)
{
    LinvRow l;
    const unsigned i = (unsigned)t >> 3, w1 = (unsigned)W - 1;
#pragma unroll
    for (unsigned k = 0; k < 4; k++) {
        const unsigned j = 2 * (t & 7) + 16 * k;
        if constexpr (FWD) {
            const unsigned o = base + (j * w1 + i) * 8u;
            l.v[k].x = __builtin_bit_cast(
                double, __builtin_amdgcn_raw_buffer_load_b64(ab, (int)(j <= i ? o : out), 0, 0));
            l.v[k].y = __builtin_bit_cast(
                double, __builtin_amdgcn_raw_buffer_load_b64(ab, (int)(j < i ? o + w1 * 8u : out), 0, 0));
        } else {
            l.v[k] = __builtin_bit_cast(
                f64x2, __builtin_amdgcn_raw_buffer_load_b128(ab, (int)(base + (i * w1 + j) * 8u), 0, 0));
        }
    }
    return l;
}
__device__ __forceinline__ double linv_times(const LinvRow &r, const double *y, int t)
{
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        s += r.v[k].x * y[2 * (t & 7) + 16 * k];
        s += r.v[k].y * y[2 * (t & 7) + 16 * k + 1];
    }
    return sum8(s);
}

// A wave's share of a panel: the 64 rows of row block rb next to solved
// block k.  Loads of a wave without a share (rb past the panel) are out of
// range and read nothing, so they need no branch.
//
// Forward, rows below: column c of the block at a + c (W - 1), lane = row.
// Backward, rows above: row i's 64 entries of the block are contiguous in
// the band, 8 rows at a time: lane = 8 (row) + p, lane p takes entries
// 2 p + 16 j (+ 1), so a load covers 128 contiguous bytes of each row.
struct Panel {
    f64x2 v[32];
};
template <bool FWD>
__device__ __forceinline__ void load_panel(__amdgpu_buffer_rsrc_t ab, int W, int k, int rb, bool mine,
                                           unsigned lane, Panel &p)
{
    const unsigned w8 = (unsigned)(W - 1) * 8u;
    unsigned o;
    if constexpr (FWD)
        o = (unsigned)k * kBandNB * (unsigned)W * 8u + kBandNB * 8u * (1u + rb) + lane * 8u;
    else
        o = ((unsigned)(k - 1 - rb) * kBandNB + (lane >> 3)) * w8 + (unsigned)k * kBandNB * 8u +
            (lane & 7) * 16u;
    o = mine ? o : ~0u - 64u * w8 - 512u;
#pragma unroll
    for (int c = 0; c < 32; c++) {
        if constexpr (FWD) {
            p.v[c].x = __builtin_bit_cast(
                double, __builtin_amdgcn_raw_buffer_load_b64(ab, (int)(o + 2 * c * w8), 0, 0));
            p.v[c].y = __builtin_bit_cast(
                double, __builtin_amdgcn_raw_buffer_load_b64(ab, (int)(o + (2 * c + 1) * w8), 0, 0));
        } else {
            p.v[c] = __builtin_bit_cast(
                f64x2, __builtin_amdgcn_raw_buffer_load_b128(
                           ab, (int)(o + (c >> 2) * 8u * w8 + (c & 3) * 128u), 0, 0));
        }
    }
}
// forward: row `lane`; backward: lane 8 r + p gets the sum of row 8 p + r
template <bool FWD>
__device__ __forceinline__ double panel_times(const Panel &p, const double *x, int lane)
{
    if constexpr (FWD) {
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int c = 0; c < 32; c++) {
            s0 += p.v[c].x * x[2 * c];
            s1 += p.v[c].y * x[2 * c + 1];
        }
        return s0 + s1;
    } else {
        f64x2 xv[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            xv[j].x = x[2 * (lane & 7) + 16 * j];
            xv[j].y = x[2 * (lane & 7) + 16 * j + 1];
        }
        double out = 0.0;
#pragma unroll
        for (int g = 0; g < 8; g++) {
            double s = 0.0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                s += p.v[4 * g + j].x * xv[j].x;
                s += p.v[4 * g + j].y * xv[j].y;
            }
            s = sum8(s);
            out = (lane & 7) == g ? s : out;
        }
        return out;
    }
}

__device__ __forceinline__ bool served(const ClassDev &C, int smp, int mode)
{
    return mode < 0 || mg_act(C.mg_st[smp], mode);
}

// The sweeps of one sample in one workgroup of 8 waves (narrow bands and
// batches of samples), in place on by.  The band window of the right-hand
// side lives in LDS (slot = block modulo the window), every wave holds 64
// rows of the current panel in registers, loaded before the diagonal product
// they wait for.  sweeps: bit 0 forward, bit 1 backward.
__device__ __forceinline__ void sweep_sample(const ClassDev &C, int smp, int sweeps,
                                             double *yw /* bW */, double *xb /* kBandNB */)
{
    const int n = C.bn, W = C.bW, nblk = (n + kBandNB - 1) / kBandNB, nwb = W / kBandNB;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    // bytes of the factor and of a block of columns
    const unsigned nw = (unsigned)n * (unsigned)W * 8u, bw = kBandNB * (unsigned)W * 8u;
    const __amdgpu_buffer_rsrc_t ab =
        wave_view(glob((const double *)C.band + (size_t)smp * C.band_ss), nw);
    GLOB double *y = glob(C.by + (size_t)smp * n);
    if (sweeps & 1) {
        for (int i = t; i < W; i += 64 * kSweepWaves) yw[i] = i < n ? y[i] : 0.0;
        LinvRow li = load_linv<true>(ab, 0, nw, W, t);
        __syncthreads();
        for (int k = 0; k < nblk; k++) {
            const int k0 = k * kBandNB, slot = (k % nwb) * kBandNB;
            const int nrb = min(nblk - 1 - k, nwb - 1);  // row blocks below
            Panel p;
            load_panel<true>(ab, W, k, wave, wave < nrb, lane, p);
            const int in = k0 + W + lane;  // the block entering the window
            const double yin = wave == kSweepWaves - 1 && in < n ? y[in] : 0.0;
            const double x = linv_times(li, yw + slot, t);
            if ((t & 7) == 0) {
                xb[t >> 3] = x;
                if (k0 + (t >> 3) < n) y[k0 + (t >> 3)] = x;
            }
            if (k + 1 < nblk) li = load_linv<true>(ab, (k + 1) * bw, nw, W, t);
            __syncthreads();
            if (wave < nrb) yw[((k + 1 + wave) % nwb) * kBandNB + lane] -= panel_times<true>(p, xb, lane);
            if (wave == kSweepWaves - 1) yw[slot + lane] = yin;
            __syncthreads();
        }
    }
    if (sweeps & 2) {
        __syncthreads();
        const int kl = nblk - 1;
        for (int j = wave; j < min(nwb, nblk); j += kSweepWaves) {
            const int i = (kl - j) * kBandNB + lane;
            yw[((kl - j) % nwb) * kBandNB + lane] = i < n ? y[i] : 0.0;
        }
        LinvRow li = load_linv<false>(ab, kl * bw, nw, W, t);
        __syncthreads();
        for (int k = kl; k >= 0; k--) {
            const int k0 = k * kBandNB, slot = (k % nwb) * kBandNB;
            const int nrb = min(k, nwb - 1);  // row blocks above
            Panel p;
            load_panel<false>(ab, W, k, wave, wave < nrb, lane, p);
            const int in = k0 - W + lane;
            const double yin = wave == kSweepWaves - 1 && in >= 0 ? y[in] : 0.0;
            const double x = linv_times(li, yw + slot, t);
            if ((t & 7) == 0) {
                xb[t >> 3] = x;
                if (k0 + (t >> 3) < n) y[k0 + (t >> 3)] = x;
            }
            if (k > 0) li = load_linv<false>(ab, (k - 1) * bw, nw, W, t);
            __syncthreads();
            if (wave < nrb)
                yw[((k - 1 - wave) % nwb) * kBandNB + (lane & 7) * 8 + (lane >> 3)] -=
                    panel_times<false>(p, xb, lane);
            if (wave == kSweepWaves - 1) yw[slot + lane] = yin;
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(64 * kSweepWaves) void k_band_sweep_one(const ClassDev *__restrict__ cp,
                                                                     int mode, int sweeps)
{
    extern __shared__ double yw[];
    __shared__ double xb[kBandNB];
    const ClassDev &C = *cp;
    const int smp = blockIdx.x;
    if (!served(C, smp, mode)) return;
    sweep_sample(C, smp, sweeps, yw, xb);
}

// Coarsest multigrid levels, all classes of the batch at once: items are
// (class, sample), one workgroup each, which also moves the level's
// right-hand side into band order and the solution back.  A sample's sweeps
// are a serial chain of 3.3 us a block and sweep, so a batch's classes one after the
// other waited for the sum of their chains instead of the longest: 17 samples
// over four meshes (coarsest chains of 53, 23 and 9 blocks) 31.1 -> 26.4 ms.
template <typename real>
__global__ __launch_bounds__(64 * kSweepWaves) void k_mg_band_solve(const ClassDev *__restrict__ cls,
                                                                    const int2 *__restrict__ items,
                                                                    int T, int mode)
{
    extern __shared__ double yw[];
    __shared__ double xb[kBandNB];
    const ClassDev &C = cls[items[blockIdx.x].x];
    const int smp = items[blockIdx.x].y, n = C.bn, t = threadIdx.x;
    if (!served(C, smp, mode)) return;
    const size_t vb = (size_t)(smp / T) * C.tile_vec + smp % T;
    GLOB double *y = glob(C.by + (size_t)smp * n);
    const GLOB real *r = glob((const real *)C.r + vb);
    GLOB real *z = glob((real *)C.z + vb);
    for (int i = t; i < n; i += 64 * kSweepWaves) y[i] = (double)r[(size_t)C.bperm[i] * T];
    __syncthreads();
    sweep_sample(C, smp, 3, yw, xb);
    __syncthreads();
    for (int row = t; row < 3 * C.nb; row += 64 * kSweepWaves) {
        const int i = C.binv[row];
        z[(size_t)row * T] = i >= 0 ? (real)y[i] : (real)0;
    }
}

// Sums of two rows spread over the two halves of a wave: lane l < 32 gets a of
// lanes l and l + 32, lane l + 32 gets b of them.
__device__ __forceinline__ double sum_halves(double a, double b)
{
    const unsigned long long ua = __builtin_bit_cast(unsigned long long, a);
    const unsigned long long ub = __builtin_bit_cast(unsigned long long, b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)ua, (unsigned)ub, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(ua >> 32), (unsigned)(ub >> 32), false, false);
    return __builtin_bit_cast(double, ((unsigned long long)hi[0] << 32) | lo[0]) +
           __builtin_bit_cast(double, ((unsigned long long)hi[1] << 32) | lo[1]);
}

// One block of a sweep over many workgroups (wide bands, where one
// workgroup cannot stream a panel fast enough): every workgroup forms the
// block's solution from the right-hand side in `src` and subtracts its
// share of 64 rows there; workgroup 0 writes the solution to `dst`, another
// buffer, since the others still read the block.  The 8 waves split the
// panel's columns (forward) or rows (backward).  Forward, loads of 16 bytes
// along the columns: 3.6 us a launch (8 samples of 12^3), 4.1 with the 8-byte
// loads of sweep_sample.
// Forward: by -> bx, backward: bx -> by.
template <bool FWD>
__global__ __launch_bounds__(64 * kSweepWaves) void k_band_sweep_step(
    const ClassDev *__restrict__ cp, int k, int mode)
{
    __shared__ double yb[kBandNB], xb[kBandNB], red[FWD ? 2 : 1][FWD ? kSweepWaves : 1][kBandNB];
    const ClassDev &C = *cp;
    const int smp = blockIdx.y;
    if (!served(C, smp, mode)) return;
    const int n = C.bn, W = C.bW, nblk = (n + kBandNB - 1) / kBandNB, nwb = W / kBandNB;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const GLOB double *AB = glob((const double *)C.band + (size_t)smp * C.band_ss);
    GLOB double *src = glob((FWD ? C.by : C.bx) + (size_t)smp * n);
    GLOB double *dst = glob((FWD ? C.bx : C.by) + (size_t)smp * n);
    const int k0 = k * kBandNB, rb = blockIdx.x;
    const bool rows = rb < (FWD ? min(nblk - 1 - k, nwb - 1) : min(k, nwb - 1));
    const unsigned nw = (unsigned)min(kBandNB, n - k0) * (unsigned)W * 8u;  // bytes of the block's columns
    const __amdgpu_buffer_rsrc_t ab = wave_view(AB + (size_t)k0 * W, nw);
    constexpr int kc = kBandNB / kSweepWaves;
    LinvRow li;
    f64x2 lc[4], pt[4];
    double ys[4];
    // Forward, a wave takes 8 columns, each half of it every other one, a lane
    // two rows: 16-byte loads along the band's columns
    const int half = lane >> 5, l2 = 2 * (lane & 31), row = l2 + half;
    const int i = FWD ? k0 + kBandNB * (1 + rb) + row
                      : k0 - kBandNB * (1 + rb) + kc * wave + (lane >> 3);
    if constexpr (FWD) {
        // right-hand sides by scalar loads (past the band's end any value:
        // there the inverse's columns read as zeros)
        const auto *sp = (__attribute__((address_space(4))) const double *)(unsigned long long)src;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int col = kc * wave + 2 * j;
            lc[j] = __builtin_bit_cast(
                f64x2, __builtin_amdgcn_raw_buffer_load_b128(
                           ab, (int)(col + half <= l2 + 1 ? (unsigned)((col + half) * (W - 1) + l2) * 8u : nw),
                           0, 0));
            const double y0 = sp[min(k0 + col, n - 1)], y1 = sp[min(k0 + col + 1, n - 1)];
            ys[j] = half ? y1 : y0;
        }
    } else {
        li = load_linv<false>(ab, 0, nw, W, t);
        if (t < kBandNB) yb[t] = k0 + t < n ? src[k0 + t] : 0.0;
    }
    if (rows) {
        const GLOB double *a = FWD ? AB + (size_t)k0 * W + kBandNB * (1 + rb) + l2 +
                                         (size_t)(kc * wave + half) * (W - 1)
                                   : AB + (size_t)i * W + (k0 - i) + 2 * (lane & 7);
#pragma unroll
        for (int j = 0; j < 4; j++) pt[j] = *(const GLOB f64x2u *)(a + (FWD ? (size_t)2 * j * (W - 1) : 16 * j));
    }
    // the block's solution: forward, row `row` in every wave, backward in xb
    double x = 0.0;
    if constexpr (FWD) {
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            a += lc[j].x * ys[j];
            b += lc[j].y * ys[j];
        }
        red[0][wave][lane] = sum_halves(a, b);
        __syncthreads();
        const auto &p = red[0];
        x = ((p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane])) +
            ((p[4][lane] + p[5][lane]) + (p[6][lane] + p[7][lane]));
        if (rb == 0 && wave == 0 && k0 + row < n) dst[k0 + row] = x;
    } else {
        __syncthreads();
        x = linv_times(li, yb, t);
        if ((t & 7) == 0) {
            xb[t >> 3] = x;
            if (rb == 0 && k0 + (t >> 3) < n) dst[k0 + (t >> 3)] = x;
        }
        __syncthreads();
    }
    if (!rows) return;  // the whole workgroup
    double s = 0.0;
    if constexpr (FWD) {
        double xs[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double x0 = lane_f64(x, 4 * wave + j), x1 = lane_f64(x, 4 * wave + j + 32);
            xs[j] = half ? x1 : x0;
        }
        double a = 0.0, b = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            a += pt[j].x * xs[j];
            b += pt[j].y * xs[j];
        }
        s = sum_halves(a, b);
        red[1][wave][lane] = s;
        __syncthreads();
        if (wave > 0 || i >= n) return;
        s = red[1][0][lane];
#pragma unroll
        for (int w = 1; w < kSweepWaves; w++) s += red[1][w][lane];
        src[i] -= s;
    } else {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            s += pt[j].x * xb[2 * (lane & 7) + 16 * j];
            s += pt[j].y * xb[2 * (lane & 7) + 16 * j + 1];
        }
        s = sum8(s);
        if ((lane & 7) == 0) src[i] -= s;
    }
}

}  // namespace

hipError_t launch_chol_block(hipStream_t s, const ClassDev *cp, int nsamp, int k0)
{
    hipLaunchKernelGGL(k_chol_block, dim3(1, nsamp), dim3(256), 0, s, cp, k0);
    return hipGetLastError();
}

hipError_t launch_chol_panel_inv(hipStream_t s, const ClassDev *cp, int nsamp, int k0, int m)
{
    if (m <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_chol_panel_inv, dim3((m + 63) / 64, nsamp), dim3(256), 0, s, cp, k0, m);
    return hipGetLastError();
}

hipError_t launch_chol_update(hipStream_t s, const ClassDev *cp, int nsamp, int k0, int m)
{
    if (m <= 0) return hipSuccess;
    const int T = (m + kBandNB - 1) / kBandNB;
    hipLaunchKernelGGL(k_chol_update_mfma, dim3(T * (T + 1) / 2, nsamp), dim3(256), 0, s, cp, k0, m);
    return hipGetLastError();
}

hipError_t launch_band_linv(hipStream_t s, const ClassDev *cp, int nsamp, int bn)
{
    if (bn <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_band_linv, dim3((bn + kBandNB - 1) / kBandNB, nsamp), dim3(256), 0, s, cp);
    return hipGetLastError();
}

hipError_t launch_band_sweep_one(hipStream_t s, const ClassDev *cp, int nsamp, int bn, int bW,
                                 int mode, int sweeps)
{
    if (bn <= 0) return hipSuccess;
    if (!band_one_launch(bn, bW)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_band_sweep_one, dim3(nsamp), dim3(64 * kSweepWaves), bW * sizeof(double), s,
                       cp, mode, sweeps);
    return hipGetLastError();
}

hipError_t launch_mg_band_solve(hipStream_t s, bool mixed, int T, const ClassDev *d_cls,
                                const int2 *items, int nitems, int max_bW, int mode)
{
    if (nitems <= 0) return hipSuccess;
    if (max_bW > kBandOneMax) return hipErrorInvalidValue;
    const dim3 grid(nitems), block(64 * kSweepWaves);
    const size_t lds = max_bW * sizeof(double);
    if (mixed)
        hipLaunchKernelGGL(k_mg_band_solve<float>, grid, block, lds, s, d_cls, items, T, mode);
    else
        hipLaunchKernelGGL(k_mg_band_solve<double>, grid, block, lds, s, d_cls, items, T, mode);
    return hipGetLastError();
}

hipError_t launch_band_sweep_step(hipStream_t s, const ClassDev *cp, int nsamp, int bn, int bW,
                                  int k, bool forward, int mode)
{
    const int nblk = (bn + kBandNB - 1) / kBandNB;
    const int nrb = std::min(forward ? nblk - 1 - k : k, bW / kBandNB - 1);
    const dim3 grid(std::max(1, nrb), nsamp);
    if (forward)
        hipLaunchKernelGGL((k_band_sweep_step<true>), grid, dim3(64 * kSweepWaves), 0, s, cp, k, mode);
    else
        hipLaunchKernelGGL((k_band_sweep_step<false>), grid, dim3(64 * kSweepWaves), 0, s, cp, k,
                           mode);
    return hipGetLastError();
}

}  // namespace msa
