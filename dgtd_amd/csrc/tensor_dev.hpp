// Device records of the matrix-free tensor-product stage (tensor_stage.hip).
#pragma once

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

}  // namespace dgtd
