// sf_internal.h -- shared definitions of the gfx950 kernels and the C ABI wrappers.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "../../include/sailfish_hip.h"

// Floating-point contraction is off for the whole library (also passed as
// -ffp-contract=off): FP64 results must match the CPU restatement bit for bit.
#pragma clang fp contract(off)

struct sf_ctx {
    int szI, szJ, szK;
    long long S2;
    const double *on_u, *om_v, *pn, *pm;
    int device;
    int q5_stride;            // mask stride of computeMomentumPred (szJ, or szI when fixed)
    // dense boundary-code fields for the fused substep (one int32 per rho point),
    // allocated by sf_ctx_set_bc_maps; see step2d_fused.hip
    int32_t *bc_zeta, *bc_ubar, *bc_vbar;
    int bc_ready;
    int bc_vel_copy;          // a velocity map copies from a neighbour (gradient boundary)
};

namespace sf {

void set_error(const char *fmt, ...);
int hip_fail(hipError_t e, const char *what);

inline int check_launch(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, what);
    return SF_OK;
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// 1 / x: IEEE division in FP64 (bitwise parity with the CPU restatement); the hardware
// reciprocal v_rcp_f32 (1 ulp) in FP32, one instruction instead of the ~10 of an IEEE
// FP32 division.  2 * recip(x) equals 2 / x exactly in FP64 (scaling by 2 is exact).
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }

// Adams-Bashforth extrapolation over baroclinic steps of the barotropic forcing of the
// coupled substep: F (ab 0), 3/2 F - 1/2 F1 (ab 1), (23/12 F - 16/12 F1) + 5/12 F2 (ab 2)
__device__ __forceinline__ double ab_extrapolate(int ab, double F, double F1, double F2)
{
    if (ab == 0) return F;
    if (ab == 1) return 1.5 * F - 0.5 * F1;
    return ((23.0 / 12.0) * F - (16.0 / 12.0) * F1) + (5.0 / 12.0) * F2;
}

constexpr int kBlock1D = 256;

// Bytes one substep must move before the fused 2D substeps write their outputs with
// streaming (non-temporal) stores: beyond the 256 MB last-level cache the next substep
// cannot re-read them from it, and streaming keeps L2 for the halo reads.  Measured on
// 2048 x 1024: plain stores faster at 264 MiB (FP32 physics), streaming faster at 352 MiB
// (FP64 reference discretisation) and 432 MiB (FP64 physics).
constexpr double kStreamingBytes = 320.0 * (1 << 20);

// compute units of an MI355X, where a rule of sizes was measured on the whole card
constexpr int kCUs = 256;
// compute units of a device, queried once per device
inline int cu_count(int device)
{
    static int cache[64];
    if (device < 0 || device >= 64) return kCUs;
    if (cache[device] == 0) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || v <= 0) v = kCUs;
        cache[device] = v;
    }
    return cache[device];
}

inline unsigned grid1d(long long n, int block = kBlock1D)
{
    return (unsigned)((n + block - 1) / block);
}

// Blocks of water columns in XCD bands.  Block b runs on XCD b % 8, each with its own L2;
// with blocks of columns dealt out in turn, the rows j-1 and j+1 that a stencil reads belong
// to other XCDs and are fetched once per XCD.  In bands XCD x takes the x-th eighth of the
// columns, so a row fetched for its own columns serves its neighbours from L2.  Measured
// (FP32, 67 MB a field, 1024 x 512 x 32): set_maxflux 66 us -> 57; FP64 700 x 400 x 32 (72 MB):
// 71 -> 60.  Where a field passes about half the last-level cache the kernels stream from
// HBM, and eight far-apart streams lose there: FP64 1024 x 512 x 32 (138 MB) 140 us -> 157,
// tracer step 503 -> 520.  So bands up to 100 MB a field.
constexpr double kBandBytes = 100e6;
inline unsigned column_grid(long long n, int block = kBlock1D) { return (grid1d(n, block) + 7) / 8 * 8; }
// The grid of `blocks` (a multiple of 16 or 8) blocks of `threads`: a launch takes fewer than
// 2^32 threads along x, so more of them go to rows of blocks (no bands there: fields of that
// size pass kBandBytes by far).
inline dim3 wide_grid(unsigned blocks, unsigned threads)
{
    unsigned y = 1;
    while ((unsigned long long)(blocks / y + 16) * threads >= (1ull << 32)) y *= 2;
    return y == 1 ? dim3(blocks) : dim3((blocks / y + 16) / 16 * 16, y);
}
__device__ __forceinline__ unsigned column_block(bool band)
{
    return band ? (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3) : blockIdx.y * gridDim.x + blockIdx.x;
}
// the same with two blocks per block of columns (grid of 2 * column_grid), one after the other
// on the same XCD
__device__ __forceinline__ unsigned column_pair_id() { return blockIdx.y * gridDim.x + blockIdx.x; }
__device__ __forceinline__ bool column_pair_second() { return (column_pair_id() >> 3) & 1; }
__device__ __forceinline__ unsigned column_pair_block(bool band)
{
    const unsigned x = column_pair_id() & 7, k = column_pair_id() >> 4;
    return band ? x * ((gridDim.x * gridDim.y) >> 4) + k : k * 8 + x;
}

// Level waves of a kernel that can split a column's levels: four, unless the columns alone
// give every SIMD (four a CU) four waves and the column is short (at most `few` levels).
// A split column repeats what belongs to the column (index division, metrics, the sums below
// a wave's levels), which a few levels do not pay for: one / four waves at 4 levels, FP64
// 3000 x 1500 set_maxflux 142 / 148 us, omega 104 / 139, pressure gradient 337 / 467, FP32
// 68 / 117, 50 / 111, 189 / 287.  Where the lines lie, FP64 1024 x 512: set_maxflux 8 levels
// 23.9 / 24.2, 16 levels 44.9 / 45.3 (700 x 400: 26.2 / 25.0); FP32 16 levels 24.4 / 24.5;
// pressure gradient 16 levels 149 / 160 (FP32 72 / 79), 24 levels 232 / 231.
inline int level_waves(const sf_ctx *c, size_t few)
{
    return c->S2 >= 4LL * 4 * kCUs * 64 && (size_t)c->szK <= few ? 1 : 4;
}

}  // namespace sf

#define SF_REQUIRE(cond, ...)                 \
    do {                                      \
        if (!(cond)) {                        \
            sf::set_error(__VA_ARGS__);       \
            return SF_ERR_ARG;                \
        }                                     \
    } while (0)
