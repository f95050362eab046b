// Device records and face numbering of the matrix-free tensor-product stage
// (tensor_stage.hip).
#pragma once

#include <cstddef>

namespace dgtd {

// Hexahedra, per element, in the operator's precision: [0..8] dr_k/dx_d
// (k-major), face f: [9+4f..12+4f] nx ny nz fscale/2, [33] 1/eps_r, [34]
// 1/mu_r, [35] sigma/eps_r (the Global operator's conductive term).
constexpr int kHexGeoDev = 36;
// Per element: [0..5] neighbour across face f or -(code+1), [6..11] the
// neighbour's face and orientation g*8 + o (the host record as built).
constexpr int kHexConnDev = 12;

// Quadrilaterals: [0..3] dr/dx dr/dy ds/dx ds/dy, edge f: [4+3f..6+3f] nx ny
// fscale/2, [16] 1/eps_r, [17] 1/mu_r, [18] sigma/eps_r.
constexpr int kQuadGeoDev = 19;
// Per element: [0..3] neighbour across edge f or -(code+1), [4..7] the
// neighbour-node table row (f*4 + g)*2 + c (the host record as built).
constexpr int kQuadConnDev = 8;

// Face f of the tensor element is axis = 0, 1, 2 at its low (0) or high (1) end.
constexpr int tensor_face_axis(int dim, int f)
{
    return dim == 3 ? (f == 0 || f == 5 ? 2 : f == 1 || f == 3 ? 1 : 0) : (f == 0 || f == 2 ? 1 : 0);
}
constexpr int tensor_face_end(int dim, int f) { return dim == 3 ? f == 2 || f == 3 || f == 5 : f == 1 || f == 2; }

// The face node of face f on its normal line through volume node (ix, iy, iz),
// order p: a face numbers its nodes along its vertex cycle (MFEM's faces).
constexpr int tensor_face_node(int dim, int p, int f, int ix, int iy, int iz)
{
    const int n1 = p + 1;
    if (dim == 3)
        return f == 0 ? ix + n1 * (p - iy)
             : f == 1 ? ix + n1 * iz
             : f == 2 ? iy + n1 * iz
             : f == 3 ? p - ix + n1 * iz
             : f == 4 ? p - iy + n1 * iz
                      : ix + n1 * iy;
    return f == 0 ? ix : f == 1 ? iy : f == 2 ? p - ix : p - iy;
}

// Whether these agree with the element's face table (fmask: the volume node of
// each face node, faces of nfp = (p + 1)^(dim - 1)).
template <typename Table>
bool tensor_faces_match(int dim, int p, const Table& fmask)
{
    const int n1 = p + 1, nfp = dim == 3 ? n1 * n1 : n1, np = nfp * n1;
    if (fmask.size() != (size_t)(2 * dim * nfp)) return false;
    for (int f = 0; f < 2 * dim; ++f)
        for (int i = 0; i < np; ++i) {
            int x[3] = {i % n1, i / n1 % n1, dim == 3 ? i / (n1 * n1) : 0};
            const int b = tensor_face_node(dim, p, f, x[0], x[1], x[2]);
            x[tensor_face_axis(dim, f)] = tensor_face_end(dim, f) * p;
            if (fmask[(size_t)f * nfp + b] != x[0] + n1 * x[1] + n1 * n1 * x[2]) return false;
        }
    return true;
}

}  // namespace dgtd
