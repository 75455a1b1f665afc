// Rates kernel of teams of waves (kernels/rates_split.hip): its generated sections and tables.
#pragma once
#include <string>
#include <vector>

#include "mechanism.hpp"

namespace combustion {

struct RatesSplit {
  int teams = 0, parts = 0;   // a block is teams × parts waves over teams × 64 states
  std::string source;         // kernel text (extern "C" `name`)
  std::vector<double> rcp_W;  // [K]
  std::vector<double> gibbs;  // [K_a][15]
};

// fast: exponentials and logarithms on the FP32 cores (CB_FORM_FAST). Mechanisms of up to 64 species.
// one_team: a team of four waves alone in its block, for mechanisms that otherwise run two.
RatesSplit rates_split(const Mechanism& m, const std::string& name, bool fast, bool one_team = false);

}  // namespace combustion
