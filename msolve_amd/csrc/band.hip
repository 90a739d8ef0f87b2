// Triangular sweeps with the band Cholesky factors (direct solver, first-
// sample preconditioner, coarsest multigrid levels): the solve half of
// SkylineMatrix2D.Factorize / Solve (SkylineMatrix2D.cs:160-212).
//
// A sweep walks the factor in blocks of kBandNB = 64 columns, and a block
// depends on the one before: the time is the number of blocks times the
// latency of one.  So the 64 x 64 diagonal blocks are inverted once per
// factorization (k_band_linv, all blocks at once), which turns each serial
// 64-step substitution into a 64 x 64 product of one parallel step, and both
// sweeps push a solved block's contribution outwards (forward: the rows
// below; backward: the rows above), so no block waits on a reduction over
// rows that another workgroup holds.
//
// Measured (MI355X, factor and all): the first-sample preconditioner on 8
// samples of 12^3 (6084 rows, width 576, 22 applications) 525 -> 37.5 ms,
// the sweeps of a 16^3 direct solve (13872 rows) 48 -> 1.6 ms, against a
// launch pair per block and sweep with 64-step substitutions.  Both sweeps
// in one launch and one workgroup take 4.5 us per block at width 576, what
// one CU can load; a launch per block 3.6 us whatever the width.  So wide
// bands take the launches (37.5 against 42 ms at width 576), and narrow ones
// the one launch, which also costs an idle multigrid cycle next to nothing
// (17 ragged samples, coarsest level of width 384: 85 against 203 ms).
#include <hip/hip_runtime.h>

#include "msa_common.hpp"

namespace msa {

namespace {

constexpr int kLinvBlock = 2 * kBandNB * kBandNB;  // doubles per inverted block: by row, by column
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

// X = L^-1 of a 64 x 64 lower triangle in LDS by 256 threads: the four
// 16 x 16 diagonal blocks by substitution (wave w, lane = column), then the
// blocks below by distance d from the diagonal, X_ij = -X_ii sum_k L_ik X_kj,
// one block per wave on the matrix cores.  v_mfma_f64_16x16x4: lane l holds
// A[l % 16][l / 16], B[l / 16][l % 16] and, in register v, D[l / 16 + 4 v]
// [l % 16], so a product's registers are the next one's B operands.
__device__ __forceinline__ void invert_lower(double (*L)[kBandNB + 1], double (*X)[kBandNB + 1],
                                             int t)
{
    const int lane = t & 63, w = t >> 6, o = 16 * w;
    for (int e = t; e < kBandNB * kBandNB; e += 256) X[e >> 6][e & 63] = 0.0;
    __syncthreads();
    if (lane < 16) {
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            double s = i == lane ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < i; k++) s -= L[o + i][o + k] * x[k];
            x[i] = s / L[o + i][o + i];
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
                    s = __builtin_amdgcn_mfma_f64_16x16x4f64(L[16 * i + r][16 * k + 4 * q + g],
                                                             X[16 * k + 4 * q + g][16 * j + r], s,
                                                             0, 0, 0);
            f64x4 p = {0, 0, 0, 0};
#pragma unroll
            for (int q = 0; q < 4; q++)
                p = __builtin_amdgcn_mfma_f64_16x16x4f64(X[16 * i + r][16 * i + 4 * q + g], s[q], p,
                                                         0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) X[16 * i + g + 4 * v][16 * j + r] = -p[v];
        }
    }
    __syncthreads();
}

// Inverse of every diagonal block of every factor: grid (block, sample).
// Columns past the band's end (a last, partial block) invert as identity.
__global__ __launch_bounds__(256) void k_band_linv(const ClassDev *__restrict__ cp)
{
    __shared__ double L[kBandNB][kBandNB + 1], X[kBandNB][kBandNB + 1];
    const ClassDev &C = *cp;
    const int t = threadIdx.x, k0 = blockIdx.x * kBandNB, smp = blockIdx.y;
    const int nk = min(kBandNB, C.bn - k0);
    const GLOB double *AB = glob(C.band + (size_t)smp * C.band_ss);
    for (int e = t; e < kBandNB * kBandNB; e += 256) {
        const int c = e >> 6, r = e & 63;
        L[r][c] = r >= c && r < nk ? AB[(size_t)(k0 + c) * C.bW + (r - c)] : (r == c ? 1.0 : 0.0);
    }
    __syncthreads();
    invert_lower(L, X, t);
    GLOB double *out = glob(C.linv + (size_t)smp * C.linv_ss + (size_t)blockIdx.x * kLinvBlock);
    for (int e = t; e < kBandNB * kBandNB; e += 256) {
        out[e] = X[e >> 6][e & 63];                      // by row
        out[kBandNB * kBandNB + e] = X[e & 63][e >> 6];  // by column
    }
}

// ------------------------------------------------------------------- sweeps

// Row `t / P` (P = threads / 64 lanes per row) of the inverted block times
// the block's right-hand side y: a thread takes 64 / P columns, the P lanes
// of a row sum by DPP.  m: the block's inverse, by row (forward) or by
// column (backward, the transpose).
struct LinvRow {
    f64x2 v[4];
};
__device__ __forceinline__ LinvRow load_linv(const GLOB double *m, int t)
{
    LinvRow r;
    const GLOB f64x2 *p = (const GLOB f64x2 *)(m + (t >> 3) * kBandNB + (t & 7) * 8);
#pragma unroll
    for (int k = 0; k < 4; k++) r.v[k] = p[k];
    return r;
}
__device__ __forceinline__ double linv_times(const LinvRow &r, const double *y, int t)
{
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        s += r.v[k].x * y[(t & 7) * 8 + 2 * k];
        s += r.v[k].y * y[(t & 7) * 8 + 2 * k + 1];
    }
    return sum8(s);
}

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

}  // namespace

// The sweeps of one sample in one workgroup of 8 waves (narrow bands and
// batches of samples), in place on by.  The band window of the right-hand
// side lives in LDS (slot = block modulo the window), every wave holds 64
// rows of the current panel in registers, loaded before the diagonal product
// they wait for.  sweeps: bit 0 forward, bit 1 backward.
__global__ __launch_bounds__(64 * kSweepWaves) void k_band_sweep_one(const ClassDev *__restrict__ cp,
                                                                     int mode, int sweeps)
{
    extern __shared__ double yw[];  // bW
    __shared__ double xb[kBandNB];
    const ClassDev &C = *cp;
    const int smp = blockIdx.x;
    if (!served(C, smp, mode)) return;
    const int n = C.bn, W = C.bW, nblk = (n + kBandNB - 1) / kBandNB, nwb = W / kBandNB;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const __amdgpu_buffer_rsrc_t ab =
        wave_view(glob((const double *)C.band + (size_t)smp * C.band_ss), (unsigned)n * (unsigned)W * 8u);
    const GLOB double *LI = glob((const double *)C.linv + (size_t)smp * C.linv_ss);
    GLOB double *y = glob(C.by + (size_t)smp * n);
    if (sweeps & 1) {
        for (int i = t; i < W; i += 64 * kSweepWaves) yw[i] = i < n ? y[i] : 0.0;
        LinvRow li = load_linv(LI, t);
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
            if (k + 1 < nblk) li = load_linv(LI + (size_t)(k + 1) * kLinvBlock, t);
            __syncthreads();
            if (wave < nrb) yw[((k + 1 + wave) % nwb) * kBandNB + lane] -= panel_times<true>(p, xb, lane);
            if (wave == kSweepWaves - 1) yw[slot + lane] = yin;
            __syncthreads();
        }
    }
    if (sweeps & 2) {
        __syncthreads();
        const int kl = nblk - 1, ow = kBandNB * kBandNB;
        for (int j = wave; j < min(nwb, nblk); j += kSweepWaves) {
            const int i = (kl - j) * kBandNB + lane;
            yw[((kl - j) % nwb) * kBandNB + lane] = i < n ? y[i] : 0.0;
        }
        LinvRow li = load_linv(LI + (size_t)kl * kLinvBlock + ow, t);
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
            if (k > 0) li = load_linv(LI + (size_t)(k - 1) * kLinvBlock + ow, t);
            __syncthreads();
            if (wave < nrb)
                yw[((k - 1 - wave) % nwb) * kBandNB + (lane & 7) * 8 + (lane >> 3)] -=
                    panel_times<false>(p, xb, lane);
            if (wave == kSweepWaves - 1) yw[slot + lane] = yin;
            __syncthreads();
        }
    }
}

// One block of a sweep over many workgroups (wide bands, where one
// workgroup cannot stream a panel fast enough): every workgroup forms the
// block's solution from the right-hand side in `src` and subtracts its
// share of 64 rows there; workgroup 0 writes the solution to `dst`, another
// buffer, since the others still read the block.  The 8 waves split the
// panel's columns (forward) or rows (backward).
// Forward: by -> bx, backward: bx -> by.
template <bool FWD>
__global__ __launch_bounds__(64 * kSweepWaves) void k_band_sweep_step(
    const ClassDev *__restrict__ cp, int k, int mode)
{
    __shared__ double yb[kBandNB], xb[kBandNB], red[FWD ? kSweepWaves : 1][kBandNB];
    const ClassDev &C = *cp;
    const int smp = blockIdx.y;
    if (!served(C, smp, mode)) return;
    const int n = C.bn, W = C.bW, nblk = (n + kBandNB - 1) / kBandNB, nwb = W / kBandNB;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const GLOB double *AB = glob((const double *)C.band + (size_t)smp * C.band_ss);
    const GLOB double *LI = glob((const double *)C.linv + (size_t)smp * C.linv_ss);
    GLOB double *src = glob((FWD ? C.by : C.bx) + (size_t)smp * n);
    GLOB double *dst = glob((FWD ? C.bx : C.by) + (size_t)smp * n);
    const int k0 = k * kBandNB, rb = blockIdx.x;
    const bool rows = rb < (FWD ? min(nblk - 1 - k, nwb - 1) : min(k, nwb - 1));
    const LinvRow li =
        load_linv(LI + (size_t)k * kLinvBlock + (FWD ? 0 : kBandNB * kBandNB), t);
    if (t < kBandNB) yb[t] = k0 + t < n ? src[k0 + t] : 0.0;
    constexpr int kc = kBandNB / kSweepWaves;
    double pv[kc];
    f64x2 pt[4];
    const int i = FWD ? k0 + kBandNB * (1 + rb) + lane
                      : k0 - kBandNB * (1 + rb) + kc * wave + (lane >> 3);
    if (rows) {
        if constexpr (FWD) {
            const GLOB double *a =
                AB + (size_t)k0 * W + (i - k0) + (size_t)(kc * wave) * (W - 1);
#pragma unroll
            for (int c = 0; c < kc; c++) pv[c] = a[(size_t)c * (W - 1)];
        } else {
            const GLOB double *a = AB + (size_t)i * W + (k0 - i) + 2 * (lane & 7);
#pragma unroll
            for (int j = 0; j < 4; j++) pt[j] = *(const GLOB f64x2u *)(a + 16 * j);
        }
    }
    __syncthreads();
    const double x = linv_times(li, yb, t);
    if ((t & 7) == 0) {
        xb[t >> 3] = x;
        if (rb == 0 && k0 + (t >> 3) < n) dst[k0 + (t >> 3)] = x;
    }
    __syncthreads();
    if (!rows) return;  // the whole workgroup
    double s = 0.0;
    if constexpr (FWD) {
#pragma unroll
        for (int c = 0; c < kc; c++) s += pv[c] * xb[kc * wave + c];
        red[wave][lane] = s;
        __syncthreads();
        if (wave > 0 || i >= n) return;
        s = red[0][lane];
#pragma unroll
        for (int w = 1; w < kSweepWaves; w++) s += red[w][lane];
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
