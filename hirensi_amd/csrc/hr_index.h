// Addresses of a node's displacements (three doubles at 3 n, n = i + NX (j + NY k)),
// shared by the HIP kernels and the host-side checks.  Plain constexpr functions:
// the HIP compiler treats them as callable on both sides.
//
// The byte offset 24 n passes 32 bits at 2^32 / 24 = 178.9 M nodes, which a context
// of 288 GB can hold (the operator kernels refuse smaller lattices than that, the kernels
// on a state vector alone do not): the plane's part is taken in 64 bits, on a
// pointer that all lanes share, the rest of it in 32.  A lattice has at least five planes
// and less than 2^32 / 9 nodes (LATTICE_NODES), so a plane's offsets fit.
#pragma once

namespace hr {

// nodes of a lattice at most: the numbering's slots (9 per node) are 32-bit
constexpr long long LATTICE_NODES = ((1ll << 32) - 2) / 9;

constexpr long long plane_doubles(int NX, int NY, int k) { return 3ll * NX * NY * k; }
constexpr unsigned in_plane_bytes(int NX, int i, int j) { return 24u * (unsigned)(i + NX * j); }

}  // namespace hr
