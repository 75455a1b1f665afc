// Sections and tables of kernels/rates_split.hip: the reactions of a mechanism divided over the waves of a team, each
// wave's share as straight-line HIP.
#include "rates_split.hpp"

#include <algorithm>
#include <array>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <set>
#include <sstream>

#include "emit.hpp"
#include "forms.hpp"

namespace combustion {

namespace {

constexpr double kLog2e = 1.4426950408889634;
// A compiler-only fence between segments: each reads the LDS values it uses instead of keeping an earlier read live.
const char* const kFence = "  asm volatile(\"\" ::: \"memory\");\n";
// Reactions per segment. A segment's LDS values are read while the segment before it computes, and its reactions are
// evaluated side by side, factor by factor. One and two reactions at a time took 5 and 1 % longer than four (53 species),
// which fill 251 of the 256 registers.
constexpr size_t kSegment = 4, kThirdBodySegment = 2;

std::string literal(double x) {
  char buf[64];
  std::snprintf(buf, sizeof buf, "%a", x);
  return buf;
}

// Text of one mechanism's reactions. Falloff's logarithms, and the power taken of them again, are to the base that the
// kernel's log_rows and pow_rows have: 2 with the FP64 polynomials, e with the FP32 cores.
class Writer {
 public:
  Writer(const Mechanism& m, bool fast) : m_(m), fast_(fast), falloff_unit_(fast ? 1. : kLog2e) {}

  // min(FLT_MAX, A T^β e^(-θ/T)) (reaction.rs:113-139) as (β·L + a/T) + ln A under one exponential, the power of T
  // nearest β outside it: the exponent's rounding error grows with its terms (with T^β in the exponent whole the rates'
  // mean error against 80 bits was 3.76e-15 of the state's largest, as it is 3.64e-15).
  struct Rate {
    double beta, a, lnA, A;
    const char* factor;  // outside the exponential, or null
    bool constant() const { return beta == 0. && a == 0.; }
  };
  Rate rate(const RateConstant& k) const {
    const double beta = k.temperature_exponent;
    struct { double above, shift; const char* factor; } const up[] = {{3.5, 4., "T4"}, {2.5, 3., "T3"}, {1.5, 2., "T2"}, {0.5, 1., "T"}};
    const char* factor = nullptr;
    double rest = beta;
    if (beta <= -1.5) factor = "rcpT2", rest = beta + 2.;
    else if (beta <= -0.5) factor = "rcpT", rest = beta + 1.;
    else
      for (const auto& p : up)
        if (beta >= p.above) {
          factor = p.factor, rest = beta - p.shift;
          break;
        }
    return {(float)rest != 0.f ? rest : 0., -k.activation_temperature, std::log(k.preexponential_factor), k.preexponential_factor, factor};
  }
  const char* log_T() const { return fast_ ? "L" : "LT"; }
  const char* rcp_T() const { return fast_ ? "rcpT" : "rT"; }
  std::string limited(const Rate& r, const std::string& e) const {
    // without a factor the FP64 exponent is bounded instead (see evaluate)
    if (!fast_ && !r.factor) return r.constant() ? literal(std::min((double)FLT_MAX, r.A)) : e;
    const std::string v = r.constant() ? literal(r.A) : e;
    return std::string("LIMIT(") + (r.factor ? std::string(r.factor) + " * " : "") + v + ")";
  }
  // One rate constant on its own.
  std::string rate_constant(const RateConstant& k) const {
    const Rate r = rate(k);
    const std::string x = sum_terms(r.beta, log_T(), r.a, rcp_T());
    return limited(r, r.constant() ? "" : (r.factor ? "exp64(" : "KF(") + x + " + " + literal(r.lnA) + ")");
  }

  // Exponents of several exponentials, evaluated together (`name`[i]).
  struct Exponents {
    std::vector<Rate> rates;          // limited above like every rate constant
    std::vector<std::string> others;  // any expression, bounded below; after the rates
    size_t add(const Rate& r) {
      rates.push_back(r);
      return rates.size() - 1;
    }
    size_t add(const std::string& x) {  // index counts from the end of the rates
      others.push_back(x);
      return others.size() - 1;
    }
  };
  std::string evaluate(const Exponents& x, const std::string& name) const {
    const size_t nr = x.rates.size(), n = nr + x.others.size();
    if (n == 0) return "";
    std::ostringstream s;
    s << "    double " << name << "[" << n << "];\n";
    auto row = [&](auto&& f) {
      for (size_t i = 0; i < nr; i++) {
        const std::string v = name + "[" + std::to_string(i) + "]";
        s << "    " << v << f(x.rates[i], v) << ";\n";
      }
    };
    if (nr) {
      row([&](const Rate& r, const std::string&) { return " = " + literal(r.a) + " * " + rcp_T(); });
      row([&](const Rate& r, const std::string&) { return " += " + literal(r.beta) + " * " + log_T(); });
      row([&](const Rate& r, const std::string&) { return " += " + literal(r.lnA); });
      for (size_t i = 0; i < nr && !fast_; i++)
        if (!x.rates[i].factor) s << "    " << name << "[" << i << "] = __builtin_fmin(LN_FLT_MAX, " << name << "[" << i << "]);\n";
    }
    for (size_t i = 0; i < x.others.size(); i++)
      s << "    " << name << "[" << nr + i << "] = " << bounded(x.others[i]) << ";\n";
    for (size_t i = 0; i < n;) {  // rows of at most 6
      const size_t left = (n - i + 5) / 6, c = (n - i + left - 1) / left;
      s << "    exp64_rows<" << c << ">(" << name << " + " << i << ");\n";
      i += c;
    }
    return s.str();
  }

  // β·L + a/T in the unit's terms, empty when both vanish
  static std::string sum_terms(double beta, const char* L, double a, const char* r) {
    std::string s;
    if (beta != 0.) s = literal(beta) + " * " + L;
    if (a != 0.) s += (s.empty() ? "" : " + ") + literal(a) + " * " + r;
    return s;
  }

  // ln k interpolated linearly in ln P between the table pressures, the end entries beyond them, entries of one
  // pressure summed (Cantera's pressure-dependent Arrhenius; no reference counterpart, yaml.rs:120,149).
  std::string plog(const Reaction& r) const {
    std::vector<std::pair<double, std::vector<RateConstant>>> levels;
    for (const PlogEntry& e : r.plog) {
      if (levels.empty() || levels.back().first != e.P) levels.push_back({e.P, {}});
      levels.back().second.push_back(e.k);
    }
    const char *L = log_T(), *rT = rcp_T();
    std::ostringstream s;
    for (size_t i = 0; i < levels.size(); i++) {
      const auto& ks = levels[i].second;
      s << "    const double l" << i << " = ";
      if (ks.size() == 1 && ks[0].preexponential_factor > 0) {
        const std::string x = sum_terms(ks[0].temperature_exponent, L, -ks[0].activation_temperature, rT);
        s << literal(std::log(ks[0].preexponential_factor)) << (x.empty() ? "" : " + ") << x;
      } else {
        s << "log64(";
        for (size_t j = 0; j < ks.size(); j++) {
          const std::string x = sum_terms(ks[j].temperature_exponent, L, -ks[j].activation_temperature, rT);
          s << (j ? " + " : "") << literal(ks[j].preexponential_factor) << " * exp64(" << (x.empty() ? "0.0" : x) << ")";
        }
        s << ")";
      }
      s << ";\n";
    }
    s << "    double lk = l" << levels.size() - 1 << ";\n";
    if (levels.size() > 1) {
      s << "    const double lP = log64(C_tot) + L + " << literal(std::log(R)) << ";\n";
      for (int i = (int)levels.size() - 2; i >= -1; i--) {
        const double edge = std::log(levels[i + 1].first);
        s << "    if (lP <= " << literal(edge) << ") lk = ";
        if (i >= 0) {
          const double lo = std::log(levels[i].first);
          s << "l" << i << " + (l" << i + 1 << " - l" << i << ") * ((lP - " << literal(lo) << ") * " << literal(1. / (edge - lo)) << ");\n";
        } else {
          s << "l0;\n";
        }
      }
    }
    s << "    double k0 = " << (fast_ ? "LIMIT(KF(lk))" : "KF(__builtin_fmax(lk, -1100.0))") << ";\n";
    return s.str();
  }

  std::string third_body(const Reaction& r, const std::string& M) const {
    std::ostringstream s;
    s << "    double " << M << " = C_tot;\n";
    for (size_t k = 0; k < m_.species.len(); k++)
      if (r.efficiencies[k] != 1.) s << "    " << M << " += " << literal(r.efficiencies[k] - 1.) << " * " << read('c', k) << ";\n";
    return s.str();
  }

  // How reactions are evaluated side by side.
  enum class Kind { Simple, ThreeBody, Falloff, Alone };
  static Kind kind(const Reaction& r) {
    if (r.model == ReactionModel::SRI || !r.plog.empty()) return Kind::Alone;
    return r.model == ReactionModel::Troe || r.model == ReactionModel::PressureModification ? Kind::Falloff
           : r.model == ReactionModel::ThreeBody                                                        ? Kind::ThreeBody
                                                                                                        : Kind::Simple;
  }
  static size_t segment_size(Kind k) { return k == Kind::Simple ? kSegment : k == Kind::Alone ? 1 : kThirdBodySegment; }

  // The forward rate constants k0, k1, .. of a segment (reaction.rs:149-205), falloff quotients included.
  std::string forward(const std::vector<const Reaction*>& rs) const {
    const size_t n = rs.size();
    std::ostringstream s;
    auto id = [](const char* v, size_t i) { return v + std::to_string(i); };
    if (kind(*rs[0]) == Kind::Alone) return alone(*rs[0]);
    for (size_t i = 0; i < n; i++)
      if (rs[i]->model >= ReactionModel::ThreeBody) s << third_body(*rs[i], id("M", i));
    if (kind(*rs[0]) != Kind::Falloff) {
      Exponents x;
      std::vector<Rate> rate_of;
      std::vector<std::string> e;
      for (const Reaction* r : rs) {
        rate_of.push_back(rate(r->rate_constant));
        e.push_back(rate_of.back().constant() ? "" : "x[" + std::to_string(x.add(rate_of.back())) + "]");
      }
      s << evaluate(x, "x");
      for (size_t i = 0; i < n; i++) {
        s << "    double " << id("k", i) << " = " << limited(rate_of[i], e[i]);
        if (rs[i]->model == ReactionModel::ThreeBody) s << " * " << id("M", i);
        s << ";\n";
      }
      return s.str();
    }
    // Falloff: both limits' exponentials and Fcent's, all independent
    Exponents x;
    std::vector<Rate> low, high;
    std::vector<std::string> low_e, high_e;
    std::vector<std::array<int, 3>> center(n);
    for (size_t i = 0; i < n; i++) {
      RateConstant k0 = rs[i]->k0, kinf = rs[i]->rate_constant;
      if (rs[i]->model == ReactionModel::Troe) {
        k0.preexponential_factor /= kinf.preexponential_factor;
        kinf.preexponential_factor = 1.;
      }
      low.push_back(rate(k0));
      high.push_back(rate(kinf));
      auto exponent = [&](const Rate& r) { return r.constant() ? "" : "x[" + std::to_string(x.add(r)) + "]"; };
      low_e.push_back(exponent(low.back()));
      high_e.push_back(exponent(high.back()));
    }
    for (size_t i = 0; i < n; i++) {
      center[i] = {-1, -1, -1};
      if (rs[i]->model != ReactionModel::Troe) continue;
      const Troe& t = rs[i]->troe;
      center[i][0] = (int)x.add("T * " + literal(-1. / t.T3));
      if (t.T1 < 1e30) center[i][1] = (int)x.add("T * " + literal(-1. / t.T1));
      if (std::isfinite(t.T2)) center[i][2] = (int)x.add("rcpT * " + literal(-t.T2));
    }
    s << evaluate(x, "x");
    size_t troes = 0;
    for (size_t i = 0; i < n; i++) {
      s << "    const double low" << i << " = " << id("M", i) << " * " << limited(low[i], low_e[i]) << ", high" << i << " = "
        << limited(high[i], high_e[i]) << ";\n";
      troes += rs[i]->model == ReactionModel::Troe;
    }
    s << "    double r[" << n << "] = {";
    for (size_t i = 0; i < n; i++)
      s << (i ? ", " : "") << (rs[i]->model == ReactionModel::Troe ? id("high", i) : id("low", i) + " + " + id("high", i)) << " + FLT_MIN_D";
    s << "};\n    rcp64_rows<" << n << ">(r);\n";
    if (troes) {
      // ln Fcent and ln Pr, then F = 10^(log Fcent / (1 + f1²)) with f1 = lp/d, and Pr/(1 + Pr): both quotients from
      // one reciprocal
      const double ln10 = std::log(10.) * falloff_unit_;
      std::vector<size_t> at;
      for (size_t i = 0; i < n; i++)
        if (rs[i]->model == ReactionModel::Troe) at.push_back(i);
      s << "    double l[" << 2 * troes << "];\n";
      for (size_t j = 0; j < troes; j++) {
        const size_t i = at[j];
        const Troe& t = rs[i]->troe;
        const bool unit = high[i].constant();
        auto e = [&](int c) { return "x[" + std::to_string(x.rates.size() + c) + "]"; };
        s << "    const double Pr" << i << " = " << id("low", i) << (unit ? "" : " * r[" + std::to_string(i) + "]") << ";\n"
          << "    l[" << 2 * j << "] = " << literal(1. - t.A) << " * " << e(center[i][0]) << " + " << literal(t.A)
          << (center[i][1] >= 0 ? " * " + e(center[i][1]) : "") << (center[i][2] >= 0 ? " + " + e(center[i][2]) : "") << ";\n"
          << "    l[" << 2 * j + 1 << "] = Pr" << i << " + FLT_MIN_D;\n";
      }
      s << "    log_rows<" << 2 * troes << ">(l);\n    double w[" << troes << "];\n";
      for (size_t j = 0; j < troes; j++) {
        const size_t i = at[j];
        const std::string lF = "l[" + std::to_string(2 * j) + "]", lPr = "l[" + std::to_string(2 * j + 1) + "]";
        s << "    const double lp" << i << " = " << lPr << " + (-0.67 * " << lF << " - " << literal(0.4 * ln10) << "), d" << i << " = -0.14 * lp"
          << i << " + (-1.27 * " << lF << " + " << literal(0.75 * ln10) << ");\n"
          << "    const double dd" << i << " = d" << i << " * d" << i << ", qa" << i << " = lp" << i << " * lp" << i << " + dd" << i << ", qb" << i
          << " = Pr" << i << " + 1.0;\n    w[" << j << "] = qa" << i << " * qb" << i << ";\n";
      }
      s << "    rcp64_rows<" << troes << ">(w);\n    double f[" << troes << "];\n";
      for (size_t j = 0; j < troes; j++) {
        const size_t i = at[j];
        s << "    f[" << j << "] = " << bounded("l[" + std::to_string(2 * j) + "] * (dd" + std::to_string(i) + " * (w[" + std::to_string(j) + "] * qb" +
                                               std::to_string(i) + "))") << ";\n";
      }
      s << "    pow_rows<" << troes << ">(f);\n";
      for (size_t j = 0; j < troes; j++) {
        const size_t i = at[j];
        s << "    double " << id("k", i) << " = " << literal(rs[i]->rate_constant.preexponential_factor) << " * " << id("high", i) << " * f[" << j
          << "] * (Pr" << i << " * (w[" << j << "] * qa" << i << "));\n";
      }
    }
    for (size_t i = 0; i < n; i++)
      if (rs[i]->model != ReactionModel::Troe)
        s << "    double " << id("k", i) << " = " << id("low", i) << " * " << id("high", i) << " * r[" << i << "];\n";
    return s.str();
  }

  // A reaction evaluated by itself: pressure-dependent Arrhenius tables, and SRI falloff in Stewart, Larson & Golden's
  // form as Cantera documents it (reaction.rs:194-203 is unimplemented).
  std::string alone(const Reaction& r) const {
    if (!r.plog.empty()) return plog(r);
    std::ostringstream s;
    const SRI& x = r.sri;
    s << third_body(r, "M") << "    const double kinf = " << rate_constant(r.rate_constant) << ";\n"
      << "    const double Pr = M * " << rate_constant(r.k0) << " * rcp64(kinf + FLT_MIN_D);\n"
      << "    const double lg = log64(Pr + FLT_MIN_D) * " << literal(1. / std::log(10.)) << ";\n"
      << "    const double X = rcp64(1.0 + lg * lg);\n"
      << "    const double base = " << literal(x.A) << " * exp64(" << bounded("rcpT * " + literal(-x.B)) << ")";
    if (x.C != 0.) s << " + exp64(" << bounded("T * " + literal(-1. / x.C)) << ")";
    s << ";\n    double k0 = " << literal(x.D) << " * exp64(" << bounded("X * log64(base)") << ");\n";
    if (x.E != 0.) s << "    k0 *= exp64(" << bounded(literal(x.E) + " * L") << ");\n";
    s << "    k0 *= kinf * Pr * rcp64(Pr + 1.0);\n";
    return s.str();
  }

  // A segment's rates of progress and their contributions to ω, factor by factor over the reactions.
  std::string reactions(const std::vector<const Reaction*>& rs, std::vector<char>& touched) const {
    const size_t K = m_.species.len(), n = rs.size();
    std::ostringstream s;
    s << "  {";
    for (const Reaction* r : rs) s << " // " << r->equation << "\n  ";
    s << forward(rs);
    std::vector<std::vector<std::string>> a(n), b(n);
    for (size_t i = 0; i < n; i++) {
      const Reaction& r = *rs[i];
      const bool back = reversible(r);
      if (back && (r.sum_net > 2 || r.sum_net < -1)) throw ast::Error("unsupported change in the number of moles: " + r.equation);
      std::vector<std::string> e, f;
      for (size_t k = 0; k < K; k++) {
        const int both = back ? std::min(r.reactants[k], r.products[k]) : 0;
        for (int c = 0; c < both; c++) s << "    k" << i << " *= " << read('c', k) << ";\n";
        for (int c = both; c < r.reactants[k]; c++) {
          a[i].push_back(read('c', k));
          if (back && k < m_.active) e.push_back(read('e', k));
        }
        for (int c = both; back && c < r.products[k]; c++) f.push_back(read('f', k));
      }
      if (!back) continue;
      // (S P0/RT)^(-Σν), then the E- and F factors in turn (their magnitudes balance)
      if (r.sum_net < 0) b[i].push_back("C0");
      for (int c = 0; c < r.sum_net; c++) b[i].push_back("rcpC0");
      for (size_t c = 0; c < std::max(e.size(), f.size()); c++) {
        if (c < f.size()) b[i].push_back(f[c]);
        if (c < e.size()) b[i].push_back(e[c]);
      }
    }
    size_t most = 0;
    for (size_t i = 0; i < n; i++) {
      s << "    double a" << i << " = k" << i << ", b" << i << " = k" << i << ";\n";
      most = std::max({most, a[i].size(), b[i].size()});
    }
    for (size_t c = 0; c < most; c++) {
      for (size_t i = 0; i < n; i++) {
        if (c < a[i].size()) s << "    a" << i << " *= " << a[i][c] << ";\n";
        if (c < b[i].size()) s << "    b" << i << " *= " << b[i][c] << ";\n";
      }
    }
    for (size_t i = 0; i < n; i++) s << "    const double q" << i << " = a" << i << (reversible(*rs[i]) ? " - b" + std::to_string(i) : "") << ";\n";
    for (size_t k = 0; k < m_.active; k++)
      for (size_t i = 0; i < n; i++) {
        const int nu = rs[i]->net[k];
        if (nu == 0) continue;
        const std::string w = "w" + std::to_string(k), q = "q" + std::to_string(i);
        const std::string v = nu == 1 || nu == -1 ? q : literal(std::abs(nu)) + " * " + q;
        if (!touched[k]) s << "    " << w << " = " << (nu < 0 ? "-" : "") << "(" << v << ");\n";
        else s << "    " << w << (nu < 0 ? " -= " : " += ") << v << ";\n";
        touched[k] = 1;
      }
    s << "  }\n";
    return s.str();
  }

  // A segment of reactions: the LDS reads it needs (into names of its own) and its text.
  struct Segment {
    std::string reads, text;
  };
  Segment segment(const std::vector<size_t>& which, std::vector<char>& touched) {
    Segment s;
    number_++;
    reads_.clear();
    std::vector<const Reaction*> rs;
    for (size_t r : which) rs.push_back(&m_.reactions[r]);
    s.text = reactions(rs, touched);
    for (const auto& [array, k] : reads_) {
      const char* macro = array == 'c' ? "C" : array == 'f' ? "F" : "EN";
      s.reads += "  const double " + name(array, k) + " = " + macro + "(" + std::to_string(k) + ");\n";
    }
    return s;
  }

  static bool reversible(const Reaction& r) { return r.model != ReactionModel::Irreversible; }

  // Instructions of a reaction, roughly: the sections are balanced by it.
  int cost(const Reaction& r) const {
    const int exponential = 17, logarithm = 24, reciprocal = 7;
    int c = exponential + 3;
    for (size_t k = 0; k < r.net.size(); k++) c += 1 + (r.net[k] != 0);
    c += r.sum_reactants + r.sum_products;
    if (r.plog.size() > 1) c += (int)r.plog.size() * 6 + logarithm + exponential;
    if (r.model >= ReactionModel::ThreeBody)
      for (double e : r.efficiencies) c += e != 1.;
    if (r.model == ReactionModel::PressureModification) c += exponential + reciprocal + 5;
    if (r.model == ReactionModel::Troe || r.model == ReactionModel::SRI) c += 5 * exponential + 2 * logarithm + 2 * reciprocal + 15;
    return c;
  }

 private:
  // An argument that the FP64 exponential needs within 2^31 (temperatures outside any use; the FP32-core exponential
  // bounds its own).
  std::string bounded(const std::string& x) const { return fast_ ? x : "__builtin_fmax(" + x + ", -1100.0)"; }

  std::string name(char array, size_t k) const { return array + std::to_string(number_) + "_" + std::to_string(k); }
  std::string read(char array, size_t k) const {
    reads_.insert({array, k});
    return name(array, k);
  }

  const Mechanism& m_;
  bool fast_;
  double falloff_unit_;
  int number_ = 0;
  mutable std::set<std::pair<char, size_t>> reads_;
};

void replace(std::string& text, const std::string& what, const std::string& with) {
  const size_t at = text.find(what);
  if (at == std::string::npos) throw ast::Error("rates_split: the kernel template has no " + what);
  text.replace(at, what.size(), with);
}

}  // namespace

RatesSplit rates_split(const Mechanism& m, const std::string& name, bool fast, bool one_team) {
  const size_t K = m.species.len(), KA = m.active;
  RatesSplit t;
  // Eight waves per CU (two per SIMD, 256 registers each): two teams of four waves where their LDS fits (up to 54
  // species with one of them inert, which take all of it), since each part pays for the shared prologue and the sums, else one team of eight.
  t.teams = (2 * KA + K) * 128 * sizeof(double) <= 160 * 1024 ? 2 : 1;
  t.parts = 8 / t.teams;
  if (one_team) t.teams = 1;
  Writer w(m, fast);
  // Sections: the longest reaction first, each to the part with the least work so far.
  const size_t R = m.reactions.size();
  std::vector<size_t> order(R);
  for (size_t r = 0; r < R; r++) order[r] = r;
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return w.cost(m.reactions[a]) > w.cost(m.reactions[b]); });
  std::vector<std::vector<size_t>> part(t.parts);
  std::vector<int> load(t.parts, 0);
  for (size_t r : order) {
    const int p = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    part[p].push_back(r);
    load[p] += w.cost(m.reactions[r]);
  }
  std::ostringstream s;
  for (size_t k = 0; k < KA; k++) s << (k ? ", w" : "  double w") << k << " = 0.0";
  s << ";\n";
  for (int p = 0; p < t.parts; p++) {
    s << (p ? "  else if" : "  if") << " (part == " << p << ") {\n";
    std::vector<char> touched(KA, 0);
    std::vector<Writer::Segment> segments;
    std::stable_sort(part[p].begin(), part[p].end(), [&](size_t a, size_t b) { return Writer::kind(m.reactions[a]) < Writer::kind(m.reactions[b]); });
    for (size_t i = 0; i < part[p].size();) {
      std::vector<size_t> which;
      const Writer::Kind kind = Writer::kind(m.reactions[part[p][i]]);
      while (i < part[p].size() && which.size() < Writer::segment_size(kind) && Writer::kind(m.reactions[part[p][i]]) == kind)
        which.push_back(part[p][i++]);
      segments.push_back(w.segment(which, touched));
    }
    if (!segments.empty()) s << segments[0].reads << kFence;
    for (size_t i = 0; i < segments.size(); i++) {
      // The older team's waves win the issue slots and would leave the younger one's to run alone at the end, one
      // instruction per five cycles: the younger goes first for its first half (5 % of the kernel's time).
      if (i == 0 && t.teams > 1) s << "  if (team) __builtin_amdgcn_s_setprio(1);\n";
      if (i == segments.size() / 2 && t.teams > 1) s << "  __builtin_amdgcn_s_setprio(0);\n";
      s << (i + 1 < segments.size() ? segments[i + 1].reads + kFence : "") << segments[i].text;
    }
    s << "  }\n";
  }
  std::ostringstream store, add;
  for (size_t k = 0; k < KA; k++) {
    store << "    row[" << k << " * COLS] = w" << k << ";\n";
    add << "    row[" << k << " * COLS] += w" << k << ";\n";
  }
  std::ostringstream head;
  head << "#define NAME " << name << "\n#define K " << K << "\n#define KA " << KA << "\n#define PARTS " << t.parts << "\n#define TEAMS " << t.teams
       << "\n#define FAST " << (fast ? 1 : 0) << "\n";
  t.source = head.str() + rates_split_source;
  replace(t.source, "@LDS_V@", std::to_string(std::max({KA * 32 * (size_t)(t.parts * t.teams), (size_t)(t.teams == 1 ? (2 * KA + K) * 64 : 0), (size_t)1024})));
  replace(t.source, "@SECTIONS@\n", s.str());
  replace(t.source, "@STORE@\n", store.str());
  replace(t.source, "@ADD@\n", add.str());
  for (size_t k = 0; k < K; k++) t.rcp_W.push_back(1. / m.species.molar_mass[k]);
  for (size_t k = 0; k < KA; k++) {
    const NASA7& n = m.species.thermodynamics[k];
    t.gibbs.push_back(std::isnan(n.temperature_split) ? INFINITY : n.temperature_split);
    for (const auto& a : n.pieces) {
      // the arrangement of reaction.rs:78
      const double g[7] = {a[0] - a[6], -a[0], -a[1] / 2., (1. / 3. - 1. / 2.) * a[2], (1. / 4. - 1. / 3.) * a[3], (1. / 5. - 1. / 4.) * a[4], a[5]};
      t.gibbs.insert(t.gibbs.end(), g, g + 7);
    }
  }
  return t;
}

}  // namespace combustion
