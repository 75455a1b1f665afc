// Sections and tables of kernels/transport_split.hip.
#include "transport_split.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <sstream>

#include "emit.hpp"

namespace combustion {

namespace {

constexpr int kWaves = 4;

std::string literal(double x) {
  char buf[64];
  std::snprintf(buf, sizeof buf, "%a", x);
  return buf;
}

void replace(std::string& text, const std::string& what, const std::string& with) {
  const size_t at = text.find(what);
  if (at == std::string::npos) throw ast::Error("transport_split: the kernel template has no " + what);
  text.replace(at, what.size(), with);
}

const char* const kFence = "  asm volatile(\"\" ::: \"memory\");\n";

// A wave's text in blocks, each block's LDS reads one block ahead of their use.
struct Blocks {
  std::vector<std::string> reads, text;
  void add(const std::string& r, const std::string& t) {
    reads.push_back(r);
    text.push_back(t);
  }
  std::string str() const {
    std::string s = reads.empty() ? "" : reads[0] + kFence;
    for (size_t i = 0; i < text.size(); i++) s += (i + 1 < text.size() ? reads[i + 1] + kFence : "") + text[i];
    return s;
  }
};

std::string per_wave(const std::vector<std::string>& sections) {
  std::string s;
  for (size_t w = 0; w < sections.size(); w++)
    s += (w ? "  else if (wave == " : "  if (wave == ") + std::to_string(w) + ") {\n" + sections[w] + "  }\n";
  return s;
}

// The pair sums of one wave in one phase: pairs (own species slot i, species j), four reciprocals at a time.
class Pairs {
 public:
  Pairs(const Polynomials& p, int wave) : p_(p), wave_(wave) {}

  // Column j against the own slots `rows` (j another wave's species, its terms added into S(j)).
  void column(size_t j, const std::vector<int>& rows) {
    const std::string n = std::to_string(j);
    open("  const double x" + n + " = X(" + n + "), s" + n + " = S(" + n + ");\n  double t" + n + " = s" + n + ";\n");
    for (int i : rows) pair(i, kWaves * i + wave_, j, "x" + n, "t" + n);
    flush();
    text_ += "  S(" + n + ") = t" + n + ";\n";
    close();
  }
  // Pairs among the own slots.
  void own(const std::vector<int>& rows) {
    open("");
    for (int a : rows)
      for (int b : rows)
        if (b < a) pair(a, kWaves * a + wave_, kWaves * b + wave_, "x[" + std::to_string(b) + "]", "g[" + std::to_string(b) + "]");
    flush();
    close();
  }
  std::string str() const { return blocks_.str(); }

 private:
  struct Pending {
    int i;
    std::string xj, sj;
    double scale;  // of the normalised fit's reciprocal
  };
  const Polynomials& p_;
  int wave_;
  std::string reads_, text_;
  std::vector<Pending> batch_;
  Blocks blocks_;

  void open(const std::string& reads) {
    reads_ = reads;
    text_.clear();
  }
  void close() { blocks_.add(reads_, text_); }

  void pair(int i, size_t k, size_t j, const std::string& xj, const std::string& sj) {
    const double* c = &p_.diffusivityITVT[(k * p_.K + j) * p_.D];
    const bool normal = c[0] != 0.;
    std::string y = normal ? "1.0" : "0.0";
    for (int d = 1; d < p_.D; d++)
      y = "__builtin_fma(" + literal(normal ? c[d] / c[0] : c[d]) + ", pw[" + std::to_string(d) + "], " + y + ")";
    if (batch_.empty()) text_ += "  {\n";
    text_ += "    const double y" + std::to_string(batch_.size()) + " = " + y + ";\n";
    batch_.push_back({i, xj, sj, normal ? 1. / c[0] : 1.});
    if (batch_.size() == 4) flush();
  }
  void flush() {
    const size_t n = batch_.size();
    if (n == 0) return;
    if (n == 1) {
      text_ += "    const double r0 = rcp64(y0);\n";
    } else if (n == 2) {
      text_ += "    const double q = rcp64(y0 * y1), r0 = q * y1, r1 = q * y0;\n";
    } else if (n == 3) {
      text_ += "    const double p = y0 * y1, q = rcp64(p * y2), h = q * y2, r0 = h * y1, r1 = h * y0, r2 = q * p;\n";
    } else {
      text_ +=
          "    const double p = y0 * y1, o = y2 * y3, q = rcp64(p * o), h = q * o, f = q * p, r0 = h * y1, r1 = h * y0, r2 = f * y3, r3 = f * "
          "y2;\n";
    }
    for (size_t b = 0; b < n; b++) {
      const Pending& e = batch_[b];
      const std::string slot = std::to_string(e.i), R = "R" + std::to_string(b);
      text_ += "    const double " + R + " = r" + std::to_string(b) + (e.scale == 1. ? "" : " * " + literal(e.scale)) + ";\n";
      text_ += "    g[" + slot + "] += " + e.xj + " * " + R + ";\n    " + e.sj + " += x[" + slot + "] * " + R + ";\n";
    }
    text_ += "  }\n";
    batch_.clear();
  }
};

}  // namespace

std::vector<long double> wilke_factor(const std::vector<double>& W) {
  const size_t K = W.size();
  auto entry = [&](size_t k, size_t j) { return 1.L / std::sqrt((long double)W[k] + (long double)W[j]); };
  std::vector<long double> rest(K);
  std::vector<std::vector<long double>> columns;
  for (size_t k = 0; k < K; k++) rest[k] = entry(k, k);
  while (columns.size() < K) {
    // the largest remainder of a diagonal entry: no entry's remainder exceeds the mean of its two diagonal ones
    size_t pivot = 0;
    for (size_t k = 1; k < K; k++)
      if (rest[k] / entry(k, k) > rest[pivot] / entry(pivot, pivot)) pivot = k;
    if (!(rest[pivot] > std::ldexp(entry(pivot, pivot), -58))) break;
    std::vector<long double> c(K);
    for (size_t k = 0; k < K; k++) {
      long double v = entry(k, pivot);
      for (const auto& done : columns) v -= done[k] * done[pivot];
      c[k] = v / std::sqrt(rest[pivot]);
    }
    for (size_t k = 0; k < K; k++) rest[k] = k == pivot ? 0.L : rest[k] - c[k] * c[k];
    columns.push_back(c);
  }
  const size_t R = columns.size();
  std::vector<long double> G(K * R);
  for (size_t k = 0; k < K; k++)
    for (size_t r = 0; r < R; r++) G[k * R + r] = columns[r][k];
  return G;
}

TransportSplit transport_split(const Mechanism& m, const Polynomials& p) {
  TransportSplit t;
  const std::vector<double>& W = m.species.molar_mass;
  const size_t K = W.size(), D = p.D;
  const std::vector<long double> G = wilke_factor(W);
  const size_t R = G.size() / K, KW = (K + kWaves - 1) / kWaves;
  auto slots = [&](int wave) {
    std::vector<int> v;
    for (size_t i = 0; kWaves * i + wave < K; i++) v.push_back((int)i);
    return v;
  };
  // sum = or += c x, the operation spelt out: which of the first two products of a sum contraction rounds depends on the
  // text around it, and this text is also part of another kernel (rates_and_transport), with the same results
  auto term = [](const std::string& sum, const std::string& c, const std::string& x, bool first) {
    return "    " + sum + " = " + (first ? c + " * " + x : "__builtin_fma(" + c + ", " + x + ", " + sum + ")") + ";\n";
  };
  std::vector<std::string> columns, rows, own, next, half;
  for (int w = 0; w < kWaves; w++) {
    // Gᵀ y_m for the columns w, w + 4, ..; four species to a block
    Blocks b;
    for (size_t j0 = 0; j0 < K; j0 += 4) {
      std::ostringstream read, text;
      for (size_t j = j0; j < std::min(K, j0 + 4); j++) {
        read << "  const double x" << j << " = X(" << j << "), u" << j << " = S(" << j << ");\n";
        text << "  { const double y1 = x" << j << " * u" << j << ", y2 = y1 * u" << j << ";\n";
        for (size_t i = 0; kWaves * i + w < R; i++) {
          const std::string c = literal((double)(G[j * R + kWaves * i + w] * std::sqrt(W[j] / 8.L)));
          for (int mth = 0; mth < 3; mth++)
            text << term("z[" + std::to_string(i) + "][" + std::to_string(mth) + "]", c, mth == 0 ? "x" + std::to_string(j) : "y" + std::to_string(mth), j == 0);
        }
        text << "  }\n";
      }
      b.add(read.str(), text.str());
    }
    columns.push_back(b.str());
    // den's moments for the own species, divided by √W_k
    Blocks r;
    for (size_t q = 0; q < R; q++) {
      std::ostringstream read, text;
      for (int mth = 0; mth < 3; mth++) read << "  const double z" << q << "_" << mth << " = S(" << 3 * q + mth << ");\n";
      for (int i : slots(w)) {
        const size_t k = kWaves * i + w;
        const std::string c = literal((double)(G[k * R + q] / std::sqrt((long double)W[k])));
        for (int mth = 0; mth < 3; mth++) text << term("d" + std::to_string(mth) + "[" + std::to_string(i) + "]", c, "z" + std::to_string(q) + "_" + std::to_string(mth), q == 0);
      }
      r.add(read.str(), text.str());
    }
    rows.push_back(r.str());
    Pairs a(p, w), c(p, w), h(p, w);
    a.own(slots(w));
    for (int i : slots((w + 1) % kWaves)) c.column(kWaves * i + (w + 1) % kWaves, slots(w));
    // waves w and w + 2 share their pairs: the first takes its lower slots against all of the other's species, the
    // second all of its slots against the first's upper ones
    const int o = (w + 2) % kWaves;
    if (w < 2) {
      std::vector<int> lower;
      for (int i : slots(w))
        if (i < (int)KW / 2) lower.push_back(i);
      for (int i : slots(o)) h.column(kWaves * i + o, lower);
    } else {
      for (int i : slots(o))
        if (i >= (int)KW / 2) h.column(kWaves * i + o, slots(w));
    }
    own.push_back(a.str());
    next.push_back(c.str());
    half.push_back(h.str());
  }
  std::ostringstream head;
  head << "#define K " << K << "\n#define R " << R << "\n#define DD " << D << "\n";
  t.source = head.str() + transport_split_source;
  replace(t.source, "@COLUMNS@\n", per_wave(columns));
  replace(t.source, "@ROWS@\n", per_wave(rows));
  replace(t.source, "@PAIRS@\n", per_wave(own) + "  __syncthreads();\n" + per_wave(next) + "  __syncthreads();\n" + per_wave(half));
  for (size_t k = 0; k < K; k++) {
    t.rcp_W.push_back(1. / W[k]);
    t.W.push_back(W[k]);
    for (size_t d = 0; d < D; d++) {
      t.fit_c.push_back(p.conductivityIVT[k * D + d]);
      t.fit_v.push_back((double)(p.VviscosityIVVT[k * D + d] / std::sqrt(std::sqrt((long double)W[k]))));
    }
  }
  return t;
}

TransportPairs transport_pairs(const Mechanism& m, const Polynomials& p) {
  TransportPairs t;
  const std::vector<double>& W = m.species.molar_mass;
  const size_t K = W.size(), D = p.D, waves = t.waves, slots = (K + waves - 1) / waves, half = slots / 2;
  const std::vector<long double> G = wilke_factor(W);
  const size_t R = G.size() / K, KC = (K + 7) / 8 * 8;
  // the two LDS arrays, the rows of the waves' partial sums in them, and fits that can be normalised
  bool fits = slots >= 4 && (2 * K - 1) * 64 * sizeof(double) <= 160 * 1024 && K > 3 * waves && 3 * R <= K && D >= 2;
  for (size_t k = 0; k < K && fits; k++)
    for (size_t j = 0; j < k; j++) fits = fits && p.diffusivityITVT[(k * K + j) * D] != 0.;
  if (!fits) return t;
  std::ostringstream head;
  head << "#define K " << K << "\n#define KA " << m.active << "\n#define R " << R << "\n#define DD " << D << "\n#define WAVES " << waves << "\n";
  t.source = head.str() + transport_pairs_source;
  for (size_t k = 0; k < K; k++) {
    t.rcp_W.push_back(1. / W[k]);
    t.W.push_back(W[k]);
    for (size_t d = 0; d < D; d++) {
      t.fit_c.push_back(p.conductivityIVT[k * D + d]);
      t.fit_v.push_back((double)(p.VviscosityIVVT[k * D + d] / std::sqrt(std::sqrt((long double)W[k]))));
    }
  }
  t.columns.assign(R * KC, 0.);
  for (size_t r = 0; r < R; r++)
    for (size_t j = 0; j < K; j++) t.columns[r * KC + j] = (double)(G[j * R + r] * std::sqrt(W[j] / 8.L));
  t.rows.assign(waves * R * slots, 0.);
  for (size_t w = 0; w < waves; w++)
    for (size_t r = 0; r < R; r++)
      for (size_t i = 0; w + waves * i < K; i++) t.rows[(w * R + r) * slots + i] = (double)(G[(w + waves * i) * R + r] / std::sqrt((long double)W[w + waves * i]));
  // pairs of the wave's slot i (species k) with species j, a slot without species giving no term
  auto pair = [&](size_t k, size_t j) {
    const double* c = k < K && j < K ? &p.diffusivityITVT[(k * K + j) * D] : nullptr;
    for (size_t d = 1; d < D; d++) t.pairs.push_back(c ? c[d] / c[0] : 0.);
    t.pairs.push_back(c ? 1. / c[0] : 0.);
  };
  for (size_t w = 0; w < waves; w++) {
    t.offset.push_back((unsigned)t.pairs.size());
    auto column = [&](size_t j, size_t n) {
      for (size_t i = 0; i < n; i++) pair(w + waves * i, j);
    };
    for (size_t a = 1; a < slots; a++)
      for (size_t b = 0; b < a; b++) pair(w + waves * a, w + waves * b);
    for (size_t phase = 1; phase < waves / 2; phase++)
      for (size_t j = (w + phase) % waves; j < K; j += waves) column(j, slots);
    if (w < waves / 2)
      for (size_t j = w + waves / 2; j < K; j += waves) column(j, half);
    else
      for (size_t j = w - waves / 2 + waves * half; j < K; j += waves) column(j, slots);
  }
  return t;
}

}  // namespace combustion
