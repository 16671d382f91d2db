/*
 * Host-side structure of the whole-GPU multifrontal LU: the static pivot
 * sequence, the frontal tree and every index the numeric kernels use.
 */
#ifndef NGMI_SPLU_TYPES_H
#define NGMI_SPLU_TYPES_H

#include <cstdint>
#include <vector>

namespace ngmi {

constexpr int SPLU_LEAF = 64;          /* nested dissection stops at this many vertices */
/* fronts up to this many unknowns are assembled and factored in LDS by one
 * workgroup (141 x 140 doubles = 154 KiB of the CU's 160) */
constexpr int SPLU_SMALL = 140;
constexpr int SPLU_NB = 64;            /* panel width of the larger fronts */
constexpr int SPLU_CG = 16;            /* columns a workgroup assembles of a larger front */
/* a front with more children than this lists, for each of its unknowns, the
 * children whose boundary holds it; one with fewer lists, for each child, where
 * the child's boundary holds each unknown (children x unknowns, read side by
 * side; the few children of a mesh's fronts) */
constexpr int SPLU_KIDS = 16;
constexpr int SPLU_MAX_FRONT = 8000;   /* a column of a front fits 64 KB of LDS */

/* what the numeric kernels need of a front, in one record, and of each of
 * its children (kid0 on): where the Schur complement starts in the store, its
 * leading dimension and size, where its boundary's part of the solves' work
 * vector, and of the indices in the parent, starts */
struct SpluFront {
    int ns, nf, nkid, nent;
    int64_t off, idx, ent, inv, kid0, cg, gk;
    int64_t up, upe;   /* up: -1 without lists by unknown */
};
struct SpluKid {
    int64_t schur, wk;
    int ld, nb;
};
/* child q (from kid0) holds an unknown at its boundary index i */
struct SpluUp {
    int q, i;
};

struct SpluSym {
    int n = 0;
    int64_t nnz = 0;
    std::vector<int> rowsrc;             /* row r of B = P A is row rowsrc[r] of A */
    int nf = 0;                          /* fronts, in postorder */
    std::vector<int> ns, nb, parent, height;
    std::vector<int64_t> off;            /* front storage offset (doubles), nf x nf column-major */
    std::vector<int64_t> idx_off;        /* index list offset, ns + nb entries */
    std::vector<int> idx;                /* unknowns: pivots, then boundary by elimination order */
    std::vector<int> rel;                /* at a boundary slot: its index in the parent's list */
    std::vector<int> kid_ptr, kids;
    /* CSC entries by front (that of the earlier eliminated unknown): source
     * entry and local position, row | column << 16; in a larger front by
     * column, cg[cg_off[f] + 2 g] = first entry (from ent_ptr[f]) of columns
     * SPLU_CG g on, cg[.. + 2 g + 1] = first (from gk_off[f]) of the children
     * with a boundary unknown among them, listed in gk */
    std::vector<int64_t> ent_ptr, cg_off, gk_off;
    std::vector<int> ent_src, cg, gk;
    std::vector<SpluFront> front;
    std::vector<SpluKid> kid;
    std::vector<uint32_t> ent_rc;
    /* at inv_off[f] + q nf + r the boundary index in child q of the front's
     * local unknown r, or -1; kept where f has few children, or is small */
    std::vector<int64_t> inv_off;
    std::vector<int> inv;
    /* where f has many: local unknown r is held by up_ent[front[f].upe + k],
     * k from up_ptr[front[f].up + r] to the next, children in order */
    std::vector<int> up_ptr;
    std::vector<SpluUp> up_ent;
    int H = 0;                           /* largest height */
    std::vector<int> lev_ptr, lev;       /* fronts by height, by size within one */
    int max_front = 0;
    int64_t store = 0, lu_nnz = 0;
    double flops = 0;
};

int splu_analyze(int n, const int64_t *Ap, const int *Ai, SpluSym &S);

}  // namespace ngmi

#endif
