// FP64 transport kernel of four waves per 64 states (kernels/transport_split.hip): its generated sections and tables.
#pragma once
#include <string>
#include <vector>

#include "builders.hpp"
#include "mechanism.hpp"

namespace combustion {

struct TransportSplit {
  std::string source;  // extern "C" transport_fp64
  std::vector<double> rcp_W, W, fit_c, fit_v;
};
TransportSplit transport_split(const Mechanism& m, const Polynomials& p);

// FP64 transport kernel of sixteen waves per 64 states for 65 to 160 species (kernels/transport_pairs.hip).
struct TransportPairs {
  std::string source;  // extern "C" transport_tiled; empty when the kernel does not take the mechanism
  int waves = 16;
  std::vector<double> rcp_W, W, fit_c, fit_v, columns, rows, pairs;
  std::vector<unsigned> offset;  // of each wave's pairs
};
TransportPairs transport_pairs(const Mechanism& m, const Polynomials& p);

// Factor G [K][R] with G Gᵀ = 1/√(W_k + W_j) to 2^-56 of every entry (pivoted Cholesky, row-major; R is its size / K).
std::vector<long double> wilke_factor(const std::vector<double>& W);

}  // namespace combustion
