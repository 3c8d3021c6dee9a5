// The padded box of a context: where a node sits in a field.  Host code too.
#pragma once
#include <hip/hip_runtime.h>

namespace astr {

constexpr int HM = 5;   // halo width, src/commvar.F90:190
constexpr int OI = 16;  // element offset of node i=0 in a row
static_assert(OI % 16 == 0, "node i = 0 starts a 128-byte line");

struct Geo {
    int n[3];    // cells per axis (nodes 0..n)
    long s[3];   // element stride per axis (s[0] = 1)
    long org;    // element offset of node (0,0,0)
};

// The layout of a box of dims cells: rows of pi elements, a multiple of 16,
// pj rows to a plane and pk planes, halos included.
inline Geo padded_geo(const int (&dims)[3], long& pi, long& pj, long& pk)
{
    Geo g;
    pi = ((OI + dims[0] + 1 + HM) + 15) / 16 * 16;
    pj = dims[1] + 1 + 2 * HM;
    pk = dims[2] + 1 + 2 * HM;
    for (int d = 0; d < 3; ++d) g.n[d] = dims[d];
    g.s[0] = 1;
    g.s[1] = pi;
    g.s[2] = pi * pj;
    g.org = OI + HM * g.s[1] + HM * g.s[2];
    return g;
}

__host__ __device__ __forceinline__ long gidx(const Geo& g, int i, int j, int k)
{
    return g.org + i + j * g.s[1] + k * g.s[2];
}

// gidx in two parts, for kernels whose workgroups stay in a plane k: the
// element of node (0,0,k) in 64 bits, the same for the whole workgroup (a
// scalar added to the field's pointer), and from there the byte offset of the
// node in 32 bits.  The whole offset takes more than 32 bits from fields of
// 4 GiB on, about 810^3 cells, which a context that runs no line sweep may
// have; a plane of that size would make a field of 11 planes 47 GB, and a
// context has some fifty.
__host__ __device__ __forceinline__ long plane_elem(const Geo& g, int k)
{
    return g.org + k * g.s[2];
}
__host__ __device__ __forceinline__ unsigned plane_byte(const Geo& g, int i, int j)
{
    return ((unsigned)j * (unsigned)g.s[1] + (unsigned)i) * 8u;
}

}  // namespace astr
