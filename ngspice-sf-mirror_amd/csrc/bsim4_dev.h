/*
 * Device-side accessors of the BSIM4 evaluation kernels (bsim4_eval.h's
 * template contract) over the record tables.
 *
 * A record is one complete set of table fields in field order
 * ([nrec][B4F__COUNT] doubles): a model card, or a model card at one
 * geometry.  The 22 fields that L, W and delvto move (B4_IFIELDS) are kept
 * per instance as well, in tiles of 64 instances ([tile][22][64]); a kernel
 * reads all of them there (NC = 22), the 12 that L and delvto move (NC =
 * 12) or none, and the others from the record.  Which fields are
 * per instance is thus known at compile time and every field is a load at a
 * constant offset.  The table it replaces held a column code per field and
 * read each field through it: a scalar load, a wait, a branch on its sign and
 * a 64-bit address before the load itself, about 125 dependent round trips in
 * series per evaluation.
 *
 * Where all 64 lanes of a wave share one record it is read with scalar loads
 * into scalar registers (RecPrm<NC, true>); else each lane reads its own
 * (RecPrm<NC, false>).
 */
#ifndef NGMI_BSIM4_DEV_H
#define NGMI_BSIM4_DEV_H

#include <array>
#include "bsim4_fields.h"
#include "ngmi_internal.h"

namespace ngmi {

/* global and constant (scalar-loadable) address spaces: pointers that come
 * out of a descriptor in memory carry neither by themselves */
#define NGMI_GLOBAL __attribute__((address_space(1)))
#define NGMI_CONST __attribute__((address_space(4)))

constexpr int B4_TILE = 64;

/* per-instance fields: what L and delvto move, then what W moves besides */
constexpr int B4_IFIELDS[] = {
    B4F_tvth0, B4F_leff, B4F_theta0vb0, B4F_vfb, B4F_vtfbphi1, B4F_vtfbphi2, B4F_thetaRout, B4F_vfbzb,
    B4F_Aechvb, B4F_Tigb, B4F_abulkCVfactor, B4F_leffCV,
    B4F_weff, B4F_rds0, B4F_weffCJ, B4F_weffCV, B4F_czbssw, B4F_czbsswg, B4F_czbdsw, B4F_czbdswg,
    B4F_cgdoP, B4F_cgsoP};
constexpr int B4_NC_LD = 12, B4_NC_GEOM = 22;
static_assert(sizeof(B4_IFIELDS) / sizeof(int) == B4_NC_GEOM, "per-instance field list");

constexpr std::array<signed char, B4F__COUNT> b4_icols()
{
    std::array<signed char, B4F__COUNT> t{};
    for (int f = 0; f < B4F__COUNT; f++) t[f] = 127;
    for (int c = 0; c < B4_NC_GEOM; c++) t[B4_IFIELDS[c]] = (signed char)c;
    return t;
}
/* instance column of each field (127: none); column c exists when c < NC */
constexpr std::array<signed char, B4F__COUNT> B4_ICOL = b4_icols();

#ifdef __HIPCC__

/* the column form of a table (B4Tab's): the lane's instance is i0 + lane, with
 * i0 the wave's.  Pointers and strides are held here: read through the
 * descriptor, they are loaded again behind every store. */
struct ColPrm {
    const NGMI_CONST int *code;
    const NGMI_GLOBAL double *col;   /* instance i0's first column */
    const NGMI_GLOBAL double *mod;   /* the lane's model's row */
    int64_t n;
    unsigned lane;
    __device__ __forceinline__ ColPrm(const B4Tab &t, int64_t i0, unsigned lane_)
        : code((const NGMI_CONST int *)t.code), col((const NGMI_GLOBAL double *)t.itab + i0),
          mod((const NGMI_GLOBAL double *)t.mtab + (int64_t)((const NGMI_GLOBAL int *)t.model_of + i0)[lane_] * t.mcols),
          n(t.n), lane(lane_)
    {
    }
    __device__ __forceinline__ double operator()(int f) const
    {
        const int c = code[f];
        return c >= 0 ? (col + (int64_t)c * n)[lane] : mod[~c];
    }
};

template <int NC, bool UNI>
struct RecPrm;

template <int NC>
struct RecPrm<NC, true> {
    const NGMI_CONST double *rec;    /* the wave's record */
    const NGMI_GLOBAL double *col;   /* the wave's tile of instance columns */
    unsigned lane;
    __device__ __forceinline__ double operator()(int f) const
    {
        const int c = B4_ICOL[f];
        return c < NC ? col[c * B4_TILE + lane] : rec[f];
    }
};

template <int NC>
struct RecPrm<NC, false> {
    const NGMI_GLOBAL double *rec;   /* the lane's record */
    const NGMI_GLOBAL double *col;
    unsigned lane;
    __device__ __forceinline__ double operator()(int f) const
    {
        const int c = B4_ICOL[f];
        return c < NC ? col[c * B4_TILE + lane] : rec[f];
    }
};

#endif

}  // namespace ngmi

#endif
