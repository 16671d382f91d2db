/*
 * BSIM4 evaluation kernels: one thread per MOSFET instance, FP64.
 *
 * Layout: every per-instance quantity is a row of an n-strided array
 * (row r of instance i at [r * n + i]), so lane i of a wavefront touches
 * consecutive doubles of each row and every load/store is coalesced.  A
 * workgroup is one wavefront, so row bases are scalar and a lane's part of
 * an address is one 32-bit offset.
 */
#include "ngmi_internal.h"
#include "bsim4_eval.h"
#include "bsim4_dev.h"

namespace ngmi {

/* states: level l row k of the wave's lane at lv[l][k * n + lane] */
struct DevState {
    NGMI_GLOBAL double *lv[3];
    int64_t n;
    unsigned lane;
    __device__ __forceinline__ double s(int l, int k) const { return (lv[l] + k * n)[lane]; }
    __device__ __forceinline__ void set(int l, int k, double v) { (lv[l] + k * n)[lane] = v; }
};

struct DevCache {
    NGMI_GLOBAL double *c_;
    int64_t n;
    unsigned lane;
    __device__ __forceinline__ double c(int k) const { return (c_ + k * n)[lane]; }
    __device__ __forceinline__ void setc(int k, double v) { (c_ + k * n)[lane] = v; }
};

struct EvalIO {
    const double *vterm;
    double *st0, *st1, *st2;
    double *cache, *stamp, *rhs;
    int *noncon;
};

template <int FL, class P>
__device__ __forceinline__ void eval_one(const P &p, const B4Ckt &ck, const EvalIO &io, int64_t n, int64_t i0,
                                         unsigned lane)
{
    DevState st{{(NGMI_GLOBAL double *)io.st0 + i0, (NGMI_GLOBAL double *)io.st1 + i0,
                 (NGMI_GLOBAL double *)io.st2 + i0}, n, lane};
    DevCache ca{(NGMI_GLOBAL double *)io.cache + i0, n, lane};
    const NGMI_GLOBAL double *vt = (const NGMI_GLOBAL double *)io.vterm + i0;
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = (vt + k * n)[lane];
    double J[B4S__COUNT], R[B4R__COUNT];
    const int nc = b4_load<FL>(p, st, ca, ck, v, J, R);
    NGMI_GLOBAL double *js = (NGMI_GLOBAL double *)io.stamp + i0, *rs = (NGMI_GLOBAL double *)io.rhs + i0;
#pragma unroll
    for (int k = 0; k < B4S__COUNT; k++) (js + k * n)[lane] = J[k];
#pragma unroll
    for (int k = 0; k < B4R__COUNT; k++) (rs + k * n)[lane] = R[k];
    ((NGMI_GLOBAL int *)io.noncon + i0)[lane] = nc;
}

/* Column form.  WAVES = wavefronts per SIMD the register allocation aims
 * for; FL >= 0: the selector word every instance shares, compiled as a
 * constant. */
template <int WAVES, int FL>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))
k_bsim4_eval_cols(B4Tab tab, B4Ckt ck, EvalIO io)
{
    const int64_t i0 = (int64_t)blockIdx.x * 64;
    const unsigned lane = threadIdx.x;
    if (i0 + lane >= tab.n) return;
    eval_one<FL>(ColPrm(tab, i0, lane), ck, io, tab.n, i0, lane);
}

/* Record form.  WAVES and FL as above.  UNI: a workgroup per item (tile of 64
 * instances, record): the tile's lanes of that record run, reading it with
 * scalar loads; a tile whose instances have several records has as many
 * items.  Else a workgroup per tile, each lane reading its own record. */
template <int WAVES, int FL, int NC, bool UNI>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES)))
k_bsim4_eval(B4Tab tab, B4Ckt ck, EvalIO io)
{
    const unsigned lane = threadIdx.x;
    int tile = blockIdx.x, r = -1;
    if constexpr (UNI) {
        const NGMI_CONST int *it = (const NGMI_CONST int *)tab.items + 2 * blockIdx.x;
        tile = it[0];
        r = it[1];
    }
    const int64_t i0 = (int64_t)tile * B4_TILE;
    const int ri = i0 + lane < tab.n ? ((const NGMI_GLOBAL int *)tab.rec_of + i0)[lane] : -1;
    const NGMI_GLOBAL double *col = (const NGMI_GLOBAL double *)tab.itile + i0 * B4_NC_GEOM;
    if constexpr (UNI) {
        if (ri != r) return;
        /* opaque, or the equality above lets the compiler address the record
         * by the lanes' copy of its index, and no load is scalar */
        asm volatile("" : "+s"(r));
        RecPrm<NC, true> p{(const NGMI_CONST double *)tab.rec + (int64_t)r * B4F__COUNT, col, lane};
        eval_one<FL>(p, ck, io, tab.n, i0, lane);
    } else {
        if (ri < 0) return;
        RecPrm<NC, false> p{(const NGMI_GLOBAL double *)tab.rec + (int64_t)ri * B4F__COUNT, col, lane};
        eval_one<FL>(p, ck, io, tab.n, i0, lane);
    }
}

int launch_bsim4_eval(const B4Tab &tab, const B4Ckt &ck, const double *vterm,
                      double *const state[3], double *cache, double *stamp, double *rhs,
                      int *noncon, hipStream_t stream)
{
    if (tab.n == 0) return NGMI_OK;
    EvalIO io{vterm, state[0], state[1], state[2], cache, stamp, rhs, noncon};
    const dim3 nb((unsigned)((tab.n + 63) / 64));
    const bool dflt = tab.flags == B4FL_DEFAULT && tune_get(TUNE_SPECIALISE);
    const unsigned wgs = tab.mode == B4T_UNIFORM ? (unsigned)tab.nitems : nb.x;
    const int waves = waves_for(TUNE_EVAL_WAVES, (int64_t)wgs * 64);
#define NGMI_EVAL(...) hipLaunchKernelGGL((k_bsim4_eval<__VA_ARGS__>), dim3(wgs), dim3(64), 0, stream, tab, ck, io)
#define NGMI_EVAL_W(...) \
    do { \
        if (waves == 1) NGMI_EVAL(1, __VA_ARGS__); \
        else NGMI_EVAL(2, __VA_ARGS__); \
    } while (0)
    if (tab.mode == B4T_COLUMNS) {
#define NGMI_COLS(W, F) hipLaunchKernelGGL((k_bsim4_eval_cols<W, F>), nb, dim3(64), 0, stream, tab, ck, io)
        if (dflt && waves == 1) NGMI_COLS(1, B4FL_DEFAULT);
        else if (dflt) NGMI_COLS(2, B4FL_DEFAULT);
        else if (waves == 1) NGMI_COLS(1, -1);
        else NGMI_COLS(2, -1);
#undef NGMI_COLS
    } else if (tab.mode == B4T_LANES) {
        if (dflt) NGMI_EVAL_W(B4FL_DEFAULT, B4_NC_GEOM, false);
        else NGMI_EVAL_W(-1, B4_NC_GEOM, false);
    } else if (!dflt) {
        NGMI_EVAL_W(-1, B4_NC_GEOM, true);
    } else if (tab.nc == 0) {
        NGMI_EVAL_W(B4FL_DEFAULT, 0, true);
    } else {
        NGMI_EVAL_W(B4FL_DEFAULT, B4_NC_GEOM, true);
    }
#undef NGMI_EVAL_W
#undef NGMI_EVAL
    NGMI_HIP(hipGetLastError());
    return NGMI_OK;
}

}  // namespace ngmi
