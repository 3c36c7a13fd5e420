// api_vision.hip -- the vision tower (src/cuda-vision.lisp): weights and driver.
#include "api_host.h"

// --- the vision tower (replaces src/cuda-vision.lisp's q3vision) ------------------------------

namespace {

// the tower's dimensions (src/host.lisp:104-112; inspect/ref_vision.py:20-22)
const int kVisD = 1152, kVisHeads = 16, kVisHd = 72, kVisF = 4304, kVisDepth = 27, kVisOut = 4096, kVisSide = 48;
const int kVisDeep[3] = {8, 16, 24};

// every tensor the tower reads, as inspect/ref_vision.py names them, row-major shapes
std::vector<VExpect> vision_expected() {
  std::vector<VExpect> r;
  const int64_t d = kVisD, f = kVisF, o = kVisOut;
  auto add = [&](const std::string& n, std::vector<int64_t> s) { r.push_back(VExpect{n, s}); };
  add("v.patch_embd.weight", {d, 3, 16, 16});
  add("v.patch_embd.weight.1", {d, 3, 16, 16});
  add("v.patch_embd.bias", {d});
  add("v.position_embd.weight", {(int64_t)kVisSide * kVisSide, d});
  char p[64];
  for (int i = 0; i < kVisDepth; ++i) {
    snprintf(p, sizeof p, "v.blk.%d.", i);
    const std::string b = p;
    add(b + "ln1.weight", {d});
    add(b + "ln1.bias", {d});
    add(b + "attn_qkv.weight", {3 * d, d});
    add(b + "attn_qkv.bias", {3 * d});
    add(b + "attn_out.weight", {d, d});
    add(b + "attn_out.bias", {d});
    add(b + "ln2.weight", {d});
    add(b + "ln2.bias", {d});
    add(b + "ffn_up.weight", {f, d});
    add(b + "ffn_up.bias", {f});
    add(b + "ffn_down.weight", {d, f});
    add(b + "ffn_down.bias", {d});
  }
  for (int j = 0; j < 3; ++j) {
    snprintf(p, sizeof p, "v.deepstack.%d.", kVisDeep[j]);
    const std::string b = p;
    add(b + "norm.weight", {4 * d});
    add(b + "norm.bias", {4 * d});
    add(b + "fc1.weight", {4 * d, 4 * d});
    add(b + "fc1.bias", {4 * d});
    add(b + "fc2.weight", {o, 4 * d});
    add(b + "fc2.bias", {o});
  }
  add("v.post_ln.weight", {d});
  add("v.post_ln.bias", {d});
  add("mm.0.weight", {4 * d, 4 * d});
  add("mm.0.bias", {4 * d});
  add("mm.2.weight", {o, 4 * d});
  add("mm.2.bias", {o});
  return r;
}

}  // namespace

// what a split product needs of a weight: the largest |x|, the largest row's 2-norm (a vector is
// one row) and, of a matrix whose values are fp16 times 2^-kw, those fp16 rows (kp apart).  Those of
// a tensor stored and not (yet) measured bound nothing: its products, and those that its bounds
// reach, run in fp32
struct VisFacts {
  double mx = INFINITY, norm = INFINITY;
  uint16_t* h = nullptr;
  int kp = 0, kw = 0;
  bool exact = false;
};

// one product of the tower: its fp32 weights and, where SPLIT, the fp16 rows and the exponents of
// its input's scale (2^ex) and of the weights'
struct VisMm {
  const float *w = nullptr, *b = nullptr;
  const uint16_t* h = nullptr;
  int n = 0, k = 0, kp = 0, kw = 0, ex = 0;
  bool split = false;
  float descale() const { return std::ldexp(1.f, -(ex + kw)); }
};
struct VisBlock {
  const float *ln1w, *ln1b, *ln2w, *ln2b;
  VisMm qkv, out, up, down;
  int eq = 0, ek = 0, ev = 0;   // the exponents of split q, k, v
  bool heads = false;           // attention on split heads
};
struct VisMerger {
  const float *lnw, *lnb;
  VisMm fc1, fc2;
};

// A block (0 .. 26) or a merger (27 ..): for each of its products, in order, the largest
// |w_j| / T_j (k_vis_rows), and q's and k's mean squares
constexpr int kVisUnits = kVisDepth + 4;
struct VisSpread {
  double mm[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
  std::vector<double> qk;
};

struct exn_vision {
  exn_ctx* ctx = nullptr;
  std::vector<VExpect> expect;
  std::map<std::string, float*> t;   // fp32 device copies
  std::map<std::string, VisFacts> facts;
  VisSpread spread[kVisUnits];
  std::vector<VisBlock> blocks;       // made from the weights when one changed
  VisMerger mergers[4];               // deepstack 0 .. 2, then the merger
  bool plan_ok = false;
  std::map<std::string, Buf> bufs;
  float* pw = nullptr;                // the two patch kernels summed
  bool pw_ok = false;
  int side = 0;                       // the position table's side
  bool trace = false;
  int64_t traced_n = 0;               // patches of the traced encode
};

static int vis_buf(exn_vision* v, const char* key, size_t bytes, float** out) {
  Buf& b = v->bufs[key];
  if (b.bytes < bytes) {
    HIPCHK(hipStreamSynchronize(v->ctx->stream));
    dev_free(b.p);
    b.p = nullptr;
    b.bytes = 0;
    TRY(dev_alloc(&b.p, bytes));
    b.bytes = bytes;
  }
  *out = (float*)b.p;
  return EXN_OK;
}

static const VExpect* vis_find(const exn_vision* v, const char* name) {
  for (auto& e : v->expect)
    if (e.name == name) return &e;
  return nullptr;
}

static const float* vis_t(const exn_vision* v, const std::string& name) {
  auto it = v->t.find(name);
  return it == v->t.end() ? nullptr : it->second;
}

// the block or merger that reads tensor NAME; -1 the patch embedding
static int vis_unit(const std::string& name) {
  int i = 0;
  if (sscanf(name.c_str(), "v.blk.%d.", &i) == 1) return i;
  if (sscanf(name.c_str(), "v.deepstack.%d.", &i) == 1) return kVisDepth + (i - kVisDeep[0]) / 8;
  return name.compare(0, 3, "mm.") == 0 || name.compare(0, 9, "v.post_ln") == 0 ? kVisUnits - 1 : -1;
}

// N fp32 values (device, DATA) into tensor NAME's device copy
static int vis_store(exn_vision* v, const std::string& name, int64_t n, const float* data) {
  VisFacts& f = v->facts[name];   // the old values' go first: what follows may fail
  f.mx = f.norm = INFINITY;
  f.exact = false;
  if (vis_unit(name) >= 0) v->spread[vis_unit(name)] = VisSpread();
  v->plan_ok = false;
  float*& p = v->t[name];
  if (!p) TRY(dev_alloc((void**)&p, (size_t)n * 4));
  HIPCHK(hipMemcpyAsync(p, data, (size_t)n * 4, hipMemcpyDeviceToDevice, v->ctx->stream));
  if (name.rfind("v.patch_embd.weight", 0) == 0) v->pw_ok = false;
  return EXN_OK;
}

// UNITS' spreads, of those whose tensors are all there.  Ends with the stream idle.
static int vis_spreads(exn_vision* v, const std::vector<int>& units) {
  hipStream_t s = v->ctx->stream;
  // a unit's doubles: 8 maxima, the outputs of its first product, then its inputs and other outputs
  constexpr int64_t kOut = 8, kIn = kOut + 4608, kOther = kIn + 4608, kUnit = kOther + 4608;
  double* buf = nullptr;
  TRY(ctx_tmp(v->ctx, units.size() * kUnit * 8, (void**)&buf));
  std::vector<int> done;
  for (int u : units) {
    double* m = buf + (int64_t)done.size() * kUnit;
    bool all = true;
    for (const VExpect& e : v->expect) all &= vis_unit(e.name) != u || vis_t(v, e.name);
    if (!all) continue;
    done.push_back(u);
    char p[32];
    if (u < kVisDepth) snprintf(p, sizeof p, "v.blk.%d.", u);
    else if (u < kVisUnits - 1) snprintf(p, sizeof p, "v.deepstack.%d.", kVisDeep[u - kVisDepth]);
    else p[0] = 0;
    const std::string b = p;
    auto square = [&](const std::string& name, int n) {
      return vis_square(s, n, vis_t(v, name + ".weight"), vis_t(v, name + ".bias"), m + kIn);
    };
    auto rows = [&](const std::string& name, const double* in, int period, int gelu, double* out, int which) {
      const VExpect* e = vis_find(v, (name + ".weight").c_str());
      return vis_rows(s, (int)e->shape[0], (int)e->shape[1], vis_t(v, name + ".weight"), in, period,
                      vis_t(v, name + ".bias"), gelu, out, m + which);
    };
    HIPCHK(tensor_stats_clear(s, (uint32_t*)m, 4));
    if (u < kVisDepth) {
      HIPCHK(square(b + "ln1", kVisD));
      HIPCHK(rows(b + "attn_qkv", m + kIn, kVisD, 0, m + kOut, 0));
      HIPCHK(rows(b + "attn_out", m + kOut + 2 * kVisD, kVisD, 0, m + kOther, 1));
      HIPCHK(square(b + "ln2", kVisD));
      HIPCHK(rows(b + "ffn_up", m + kIn, kVisD, 1, m + kOther, 2));
      HIPCHK(rows(b + "ffn_down", m + kOther, kVisF, 0, m + kIn, 3));
    } else {
      const bool last = u == kVisUnits - 1;
      const int width = last ? kVisD : 4 * kVisD;
      HIPCHK(square(last ? "v.post_ln" : b + "norm", width));
      HIPCHK(rows(last ? "mm.0" : b + "fc1", m + kIn, width, 1, m + kOther, 0));
      HIPCHK(rows(last ? "mm.2" : b + "fc2", m + kOther, 4 * kVisD, 0, m + kOut, 1));
    }
  }
  std::vector<double> host(done.size() * (size_t)(8 + 2 * kVisD));
  for (size_t i = 0; i < done.size(); ++i)
    HIPCHK(hipMemcpyAsync(&host[i * (8 + 2 * kVisD)], buf + (int64_t)i * kUnit, (8 + 2 * kVisD) * 8, hipMemcpyDeviceToHost, s));
  HIPCHK(hipStreamSynchronize(s));
  for (size_t i = 0; i < done.size(); ++i) {
    const double* m = &host[i * (8 + 2 * kVisD)];
    VisSpread& r = v->spread[done[i]];
    for (int k = 0; k < 4; ++k) r.mm[k] = std::sqrt(m[k]);
    r.qk.assign(m + 8, m + 8 + 2 * kVisD);
  }
  return EXN_OK;
}

// the facts of the stored tensors WHICH (indices of expect): two passes over each on the device,
// the second, where the values fit, the fp16 rows; then their units' spreads.  Ends with the stream
// idle.
static int vis_measure(exn_vision* v, const std::vector<size_t>& which) {
  hipStream_t s = v->ctx->stream;
  float* recp = nullptr;
  TRY(vis_buf(v, "facts", v->expect.size() * 16, &recp));
  uint32_t* rec = (uint32_t*)recp;
  std::vector<uint32_t> host(which.size() * 4);
  std::vector<bool> packed(which.size(), false);   // exact only once the flag has come back
  auto dims = [&](size_t i, int64_t& rows, int64_t& cols) {
    const std::vector<int64_t>& d = v->expect[i].shape;
    rows = d.size() > 1 ? d[0] : 1;
    cols = 1;
    for (size_t k = d.size() > 1 ? 1 : 0; k < d.size(); ++k) cols *= d[k];
  };
  // the patch kernels (their input has no bound) and the position table stay fp32
  auto used = [&](size_t i) { return v->expect[i].name.compare(0, 7, "v.patch") && v->expect[i].name.compare(0, 7, "v.posit"); };
  auto fetch = [&]() -> int {
    HIPCHK(hipMemcpyAsync(host.data(), rec, host.size() * 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    return EXN_OK;
  };
  int64_t rows, cols;
  HIPCHK(tensor_stats_clear(s, rec, (int64_t)which.size()));
  for (size_t j = 0; j < which.size(); ++j)
    if (used(which[j])) {
      dims(which[j], rows, cols);
      HIPCHK(vis_stats(s, rows, cols, v->t[v->expect[which[j]].name], rec + 4 * j));
    }
  TRY(fetch());
  for (size_t j = 0; j < which.size(); ++j) {
    if (!used(which[j])) continue;
    const VExpect& e = v->expect[which[j]];
    VisFacts& f = v->facts[e.name];
    float mx;
    double ss;
    memcpy(&mx, &host[4 * j], 4);
    memcpy(&ss, &host[4 * j + 2], 8);
    f.mx = mx;
    f.norm = std::sqrt(ss) * 1.001;   // the sum's own rounding
    if (e.shape.size() < 2 || !std::isfinite(mx)) continue;
    dims(which[j], rows, cols);
    f.kp = (int)((cols + 63) / 64 * 64);
    f.kw = mx > 0.f ? std::min(40, std::max(0, 14 - std::ilogb(mx))) : 0;
    if (!f.h && dev_alloc((void**)&f.h, (size_t)((rows + 63) / 64 * 64) * f.kp * 2) != EXN_OK) continue;   // the fp32 product then
    packed[j] = true;
    HIPCHK(vis_pack(s, rows, (int)cols, f.kp, std::ldexp(1.f, f.kw), v->t[e.name], f.h, rec + 4 * j + 1));
  }
  TRY(fetch());
  for (size_t j = 0; j < which.size(); ++j)
    if (packed[j]) v->facts[v->expect[which[j]].name].exact = host[4 * j + 1] == 0;
  std::vector<int> units;
  for (size_t i : which) {
    const int u = vis_unit(v->expect[i].name);
    if (u >= 0 && std::find(units.begin(), units.end(), u) == units.end()) units.push_back(u);
  }
  return vis_spreads(v, units);
}

// the exponent that scales values of at most BOUND to between 2^14 and 2^15; false where there is
// none that the scales, their products and inverses hold as normal fp32 numbers
static bool vis_exponent(double bound, int& e) {
  if (!(bound >= 0.0) || !std::isfinite(bound)) return false;
  e = bound > 0.0 ? 14 - std::ilogb(bound * 1.01) : 0;
  return e >= -60 && e <= 60;
}

// A split value is off by up to 2^-40 of the bound B that its scale was made for, whatever its own
// size, so that a product's output j is off by up to about 2^-40 B |w_j|, and where B is far above
// what most inputs have (one LayerNorm gain or weight row far above the others, taken back by the
// next matrix's column) that passes fp32's own rounding.  Split where it is at most 2^-23 of every
// output's own size T_j: B |w_j| / T_j up to 2^17.  Of 1152 inputs one 2^12 times the others, at that
// limit: rounded to the split's parts a product is 1.4e-7 off, its fp32 sums 3.1e-7; 2^16 times: 2.2e-6.
// Normally distributed weights stand at 2^6.
constexpr double kVisSpread = 1 << 17;
// attention's output may be as small as its values over 64, where 4096 patches weigh alike
constexpr double kVisSpreadAtt = kVisSpread / 64;

// the same of a score, sum q k over a head: its error against its own size, or against 1 where it is
// smaller (exp2's input)
static bool vis_heads_fit(const std::vector<double>& qk, double bq, double bk) {
  if (qk.empty()) return false;
  const double qs = 1.4426950408889634 / std::sqrt((double)kVisHd);
  for (int h = 0; h < kVisHeads; ++h) {
    double q2 = 0, k2 = 0, s2 = 0;
    for (int d = 0; d < kVisHd; ++d) {
      const int at = h * kVisHd + d, to = h * kVisHd + (d + kVisHd / 2) % kVisHd;   // the rotary turns the two into each other
      const double q = 0.5 * (qk[at] + qk[to]) * qs * qs, k = 0.5 * (qk[kVisD + at] + qk[kVisD + to]);
      q2 += q;
      k2 += k;
      s2 += q * k;
    }
    if (!(bq * std::sqrt(k2) + bk * std::sqrt(q2) <= kVisSpread * std::max(1.0, std::sqrt(s2)))) return false;
  }
  return true;
}

// The products of the tower and, from the weights alone, which of them run split and at which
// scales.  LayerNorm's output is at most sqrt(D) max|g| + max|b| (no centred row has an element
// above sqrt(D) of its deviation), its row norm at most sqrt(D) max|g| + |b|; a product's output
// at most that norm times the largest weight row's plus max|bias|; the rotary at most sqrt(2)
// times its input; attention's output and GELU's at most their input.
static void vis_plan(exn_vision* v) {
  auto facts = [&](const std::string& n) -> const VisFacts& { return v->facts[n]; };
  auto mm = [&](const std::string& name) {
    VisMm r;
    const VExpect* e = vis_find(v, (name + ".weight").c_str());
    r.n = (int)e->shape[0];
    r.k = (int)e->shape[1];
    r.w = vis_t(v, name + ".weight");
    r.b = vis_t(v, name + ".bias");
    const VisFacts& f = facts(name + ".weight");
    r.h = f.h;
    r.kp = f.kp;
    r.kw = f.kw;
    r.split = f.exact;
    return r;
  };
  // LN's bounds on an element and on a row's norm, from its tensors and its width
  struct Bound { double el, norm; };
  auto ln = [&](const std::string& name, int width) {
    const VisFacts &g = facts(name + ".weight"), &b = facts(name + ".bias");
    const double r = std::sqrt((double)width) * g.mx;
    return Bound{r + b.mx, r + b.norm};
  };
  auto out = [&](const std::string& name, double norm) { return norm * facts(name + ".weight").norm + facts(name + ".bias").mx; };
  auto merger = [&](const std::string& norm, const std::string& fc1, const std::string& fc2, int width, const VisSpread& sp) {
    VisMerger m;
    m.lnw = vis_t(v, norm + ".weight");
    m.lnb = vis_t(v, norm + ".bias");
    m.fc1 = mm(fc1);
    m.fc2 = mm(fc2);
    const Bound z = ln(norm, width);
    const double rn = z.norm * std::sqrt(m.fc1.k / (double)width);   // the row is k / width normed ones
    const bool ok = m.fc1.split && m.fc2.split && vis_exponent(z.el, m.fc1.ex) && vis_exponent(out(fc1, rn), m.fc2.ex) &&
                    z.el * sp.mm[0] <= kVisSpread && out(fc1, rn) * sp.mm[1] <= kVisSpread;
    m.fc1.split = m.fc2.split = ok;
    return m;
  };
  v->blocks.clear();
  char p[64];
  for (int i = 0; i < kVisDepth; ++i) {
    snprintf(p, sizeof p, "v.blk.%d.", i);
    const std::string b = p;
    VisBlock k;
    k.ln1w = vis_t(v, b + "ln1.weight");
    k.ln1b = vis_t(v, b + "ln1.bias");
    k.ln2w = vis_t(v, b + "ln2.weight");
    k.ln2b = vis_t(v, b + "ln2.bias");
    k.qkv = mm(b + "attn_qkv");
    k.out = mm(b + "attn_out");
    k.up = mm(b + "ffn_up");
    k.down = mm(b + "ffn_down");
    const Bound z1 = ln(b + "ln1", kVisD), z2 = ln(b + "ln2", kVisD);
    const VisSpread& sp = v->spread[i];
    const double head = out(b + "attn_qkv", z1.norm), up = out(b + "ffn_up", z2.norm);
    const double bq = head * 1.4143 * 1.4427 / std::sqrt((double)kVisHd), bk = head * 1.4143;
    k.qkv.split = k.qkv.split && vis_exponent(z1.el, k.qkv.ex) && z1.el * sp.mm[0] <= kVisSpread;
    // V's parts are averaged as V is, so that they ask what attn_out asks of the averages
    k.heads = vis_exponent(bq, k.eq) && vis_exponent(bk, k.ek) && vis_exponent(head, k.ev) &&
              vis_heads_fit(sp.qk, bq, bk) && head * sp.mm[1] <= kVisSpread;
    k.out.ex = k.ev;
    k.out.split = k.out.split && k.heads && head * sp.mm[1] <= kVisSpreadAtt;
    const bool ok = k.up.split && k.down.split && vis_exponent(z2.el, k.up.ex) && vis_exponent(up, k.down.ex) &&
                    z2.el * sp.mm[2] <= kVisSpread && up * sp.mm[3] <= kVisSpread;
    k.up.split = k.down.split = ok;
    v->blocks.push_back(k);
  }
  for (int j = 0; j < 3; ++j) {
    snprintf(p, sizeof p, "v.deepstack.%d", kVisDeep[j]);
    const std::string b = p;
    v->mergers[j] = merger(b + ".norm", b + ".fc1", b + ".fc2", 4 * kVisD, v->spread[kVisDepth + j]);
  }
  v->mergers[3] = merger("v.post_ln", "mm.0", "mm.2", kVisD, v->spread[kVisUnits - 1]);
  v->plan_ok = true;
}


int exn_vision_create(exn_ctx* ctx, exn_vision** out) {
  TRY(use(ctx));
  if (!out) FAIL(EXN_EINVAL, "null output");
  exn_vision* v = new exn_vision();
  v->ctx = ctx;
  v->expect = vision_expected();
  *out = v;
  return EXN_OK;
}

int exn_vision_release(exn_vision* v) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  TRY(use(v->ctx));
  HIPCHK(hipStreamSynchronize(v->ctx->stream));
  for (auto& kv : v->bufs) dev_free(kv.second.p);
  v->bufs.clear();
  v->traced_n = 0;
  return EXN_OK;
}

int exn_vision_destroy(exn_vision* v) {
  if (!v) return EXN_OK;
  TRY(exn_vision_release(v));
  for (auto& kv : v->t) dev_free(kv.second);
  for (auto& kv : v->facts) dev_free(kv.second.h);
  dev_free(v->pw);
  delete v;
  return EXN_OK;
}

int exn_vision_set(exn_vision* v, const char* name, int kind, const void* data, const int64_t* dims, int ndims) {
  if (!v || !name || !data || !dims) FAIL(EXN_EINVAL, "vision set: null argument");
  TRY(use(v->ctx));
  const VExpect* e = vis_find(v, name);
  if (!e) FAIL(EXN_EINVAL, "vision set: no tower tensor %s", name);
  if (kind != EXN_F32 && kind != EXN_F16 && kind != EXN_BF16)
    FAIL(EXN_EINVAL, "vision set %s: kind %d (F32, F16 or BF16 only)", name, kind);
  const bool table = e->name == "v.position_embd.weight";
  bool same = ndims == (int)e->shape.size();
  for (int i = 0; same && i < ndims; ++i) same = dims[i] == e->shape[i] || (table && i == 0);
  int side = 0;
  if (same && table) {
    side = (int)std::lround(std::sqrt((double)dims[0]));
    same = side >= 2 && (int64_t)side * side == dims[0];
  }
  if (!same) {
    std::string want;
    for (auto d : e->shape) want += (want.empty() ? "" : " ") + std::to_string(d);
    FAIL(EXN_EINVAL, "vision set %s: shape is not (%s)%s", name, want.c_str(), table ? ", S square" : "");
  }
  int64_t n = 1;
  for (int i = 0; i < ndims; ++i) n *= dims[i];
  if (table && v->t.count(e->name) && v->side != side) {
    HIPCHK(hipStreamSynchronize(v->ctx->stream));
    dev_free(v->t[e->name]);
    v->t.erase(e->name);
  }
  float* tmp = nullptr;
  TRY(ctx_tmp(v->ctx, (size_t)n * 6, (void**)&tmp));   // fp32 values, and behind them the 16-bit ones as given
  if (kind == EXN_F32) {
    HIPCHK(hipMemcpyAsync(tmp, data, (size_t)n * 4, hipMemcpyHostToDevice, v->ctx->stream));
  } else {
    uint16_t* raw = (uint16_t*)(tmp + n);
    HIPCHK(hipMemcpyAsync(raw, data, (size_t)n * 2, hipMemcpyHostToDevice, v->ctx->stream));
    HIPCHK(vis_widen(v->ctx->stream, n, raw, kind == EXN_BF16, tmp));
  }
  TRY(vis_store(v, e->name, n, tmp));
  if (table) v->side = side;
  return vis_measure(v, {(size_t)(e - v->expect.data())});
}

// every tower tensor from the counter generator (the oracle's SynthVision): value = base +
// scale * normal i of key(seed, 6000 + the tensor's index), matrices then rounded to fp16
int exn_vision_synth(exn_vision* v, uint64_t seed) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  TRY(use(v->ctx));
  for (size_t i = 0; i < v->expect.size(); ++i) {
    const VExpect& e = v->expect[i];
    const std::string& nm = e.name;
    int64_t n = 1;
    for (auto d : e.shape) n *= d;
    double base = 0.0, scale;
    bool f16 = true;
    if (e.shape.size() == 1) {
      f16 = false;
      const bool bias = nm.size() > 5 && nm.compare(nm.size() - 5, 5, ".bias") == 0;
      base = bias ? 0.0 : 1.0;
      scale = bias ? 0.02 : 0.1;
    } else if (nm == "v.position_embd.weight") {
      scale = 1.0;
    } else {
      int64_t fan = 1;
      for (size_t k = 1; k < e.shape.size(); ++k) fan *= e.shape[k];
      auto ends = [&](const char* s) { return nm.size() >= strlen(s) && nm.compare(nm.size() - strlen(s), strlen(s), s) == 0; };
      double g = 1.0;
      if (nm.rfind("v.patch_embd", 0) == 0) g = 0.7;
      else if (ends("attn_qkv.weight")) g = 2.0;
      else if (ends("attn_out.weight") || ends("ffn_down.weight")) g = 0.5;
      scale = g / sqrt((double)fan);
    }
    float* tmp = nullptr;
    TRY(ctx_tmp(v->ctx, (size_t)n * 4, (void**)&tmp));
    HIPCHK(synth_normal(v->ctx->stream, gen_key(seed, 6000 + i), n, (float)base, (float)scale, 1, tmp));
    if (f16) HIPCHK(round_f16(v->ctx->stream, n, tmp));
    if (nm == "v.position_embd.weight" && v->t.count(nm) && v->side != kVisSide) {
      HIPCHK(hipStreamSynchronize(v->ctx->stream));
      dev_free(v->t[nm]);
      v->t.erase(nm);
    }
    TRY(vis_store(v, nm, n, tmp));
    if (nm == "v.position_embd.weight") v->side = kVisSide;
  }
  std::vector<size_t> all(v->expect.size());
  for (size_t i = 0; i < all.size(); ++i) all[i] = i;
  return vis_measure(v, all);
}

int exn_vision_check(exn_vision* v) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  for (auto& e : v->expect)
    if (!vis_t(v, e.name)) FAIL(EXN_ESTATE, "vision tower: missing %s", e.name.c_str());
  return EXN_OK;
}

int exn_vision_memory(exn_vision* v, int64_t* weights, int64_t* scratch_bytes) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  int64_t w = 0, s = 0;
  for (auto& e : v->expect) {
    if (!vis_t(v, e.name)) continue;
    int64_t n = 1;
    for (auto d : e.shape) n *= d;
    if (e.name == "v.position_embd.weight") n = (int64_t)v->side * v->side * kVisD;
    w += n * 4;
    auto f = v->facts.find(e.name);
    if (f != v->facts.end() && f->second.h) w += (e.shape[0] + 63) / 64 * 64 * f->second.kp * 2;
  }
  if (v->pw) w += (int64_t)kVisD * 768 * 4;
  for (auto& kv : v->bufs) s += (int64_t)kv.second.bytes;
  if (weights) *weights = w;
  if (scratch_bytes) *scratch_bytes = s;
  return EXN_OK;
}

int exn_vision_trace(exn_vision* v, int on) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  v->trace = on != 0;
  return EXN_OK;
}


// LayerNorm rows (N of WIDTH) of X, first X += BIAS + S parts where a split product left them,
// into OUT as the product NEXT reads it: split rows or fp32
static int vis_norm(exn_vision* v, int64_t n, int width, float* x, int S, const float* part, const float* bias,
                    const float* w, const float* b, const VisMm& next, float* out) {
  HIPCHK(vis_ln_s(v->ctx->stream, n, width, width, x, S, part, bias, w, b, std::ldexp(1.f, next.ex),
                  next.split ? (uint16_t*)out : nullptr, next.split ? nullptr : out));
  return EXN_OK;
}

// X (M rows, as vis_norm or the product before left them) through MM into fp32 Y, + R
static int vis_mm(exn_vision* v, const VisMm& mm, const float* x, const float* r, float* y, int64_t m) {
  hipStream_t s = v->ctx->stream;
  if (mm.split)
    HIPCHK(vis_gemm_s(s, (const uint16_t*)x, mm.h, mm.b, r, y, nullptr, m, mm.n, mm.kp, mm.descale(), 0.f, 0, 0));
  else
    HIPCHK(vis_gemm(s, x, mm.w, mm.b, r, y, m, mm.n, mm.k, 0));
  return EXN_OK;
}

// ... and GELU (ACT), as the product NEXT reads it
static int vis_mm_gelu(exn_vision* v, const VisMm& mm, const VisMm& next, const float* x, float* y, int64_t m, int act) {
  hipStream_t s = v->ctx->stream;
  if (mm.split)
    HIPCHK(vis_gemm_s(s, (const uint16_t*)x, mm.h, mm.b, nullptr, nullptr, (uint16_t*)y, m, mm.n, mm.kp, mm.descale(),
                      std::ldexp(1.f, next.ex), next.kp, act));
  else
    HIPCHK(vis_gemm(s, x, mm.w, mm.b, nullptr, y, m, mm.n, mm.k, act));
  return EXN_OK;
}

// X += X's product MM: whole, or its S parts left in PART for the next vis_norm
static int vis_mm_add(exn_vision* v, const VisMm& mm, const float* in, float* x, int64_t m, int& S, float* part) {
  S = mm.split ? vis_split(m, mm.n, mm.kp) : 1;
  if (S > 1) {
    HIPCHK(vis_gemm_part(v->ctx->stream, (const uint16_t*)in, mm.h, part, m, mm.n, mm.kp, mm.descale(), S));
    return EXN_OK;
  }
  S = 0;
  return vis_mm(v, mm, in, x, x, m);
}

// a merger (src/cuda-vision.lisp:71-82; inspect/ref_vision.py:109-118): four patches' rows as
// one row of 4608, LayerNorm after (deepstack) or before (v.post_ln, MG 3; S, PART and BIAS as
// vis_norm), fc1, GELU (erf), fc2 into OUT (M x 4096)
static int vis_merger(exn_vision* v, float* x, int n, int S, const float* part, const float* bias, float* out, int mg) {
  const int m = n / 4, d4 = 4 * kVisD;
  const VisMerger& g = v->mergers[mg];
  float *t1, *t2;
  TRY(vis_buf(v, "mt1", (size_t)n * kVisD * 4, &t1));
  TRY(vis_buf(v, "mt2", (size_t)m * d4 * 4, &t2));
  if (mg < 3) TRY(vis_norm(v, m, d4, x, S, part, bias, g.lnw, g.lnb, g.fc1, t1));
  else TRY(vis_norm(v, n, kVisD, x, S, part, bias, g.lnw, g.lnb, g.fc1, t1));
  TRY(vis_mm_gelu(v, g.fc1, g.fc2, t1, t2, m, 2));
  return vis_mm(v, g.fc2, t2, nullptr, out, m);
}

// vision-encode on the device (src/cuda-vision.lisp:34-101)
static int vis_encode(exn_vision* v, const float* px, int h, int w, float* merged, float* deep) {
  hipStream_t s = v->ctx->stream;
  const int gh = h / 16, gw = w / 16, n = gh * gw, m = n / 4, D = kVisD, np = (n + 63) / 64 * 64;
  if (!v->pw_ok) {
    if (!v->pw) TRY(dev_alloc((void**)&v->pw, (size_t)D * 768 * 4));
    HIPCHK(vis_sum(s, (int64_t)D * 768, vis_t(v, "v.patch_embd.weight"), vis_t(v, "v.patch_embd.weight.1"), v->pw));
    v->pw_ok = true;
  }
  if (!v->plan_ok) vis_plan(v);
  float *pat, *pe, *cs, *x, *hb, *qkv, *q, *k, *vt, *att, *up, *part = nullptr;
  TRY(vis_buf(v, "pat", (size_t)n * 768 * 4, &pat));
  TRY(vis_buf(v, "pe", (size_t)n * D * 4, &pe));
  TRY(vis_buf(v, "cs", (size_t)n * 144 * 4, &cs));
  TRY(vis_buf(v, "x", (size_t)n * D * 4, &x));
  TRY(vis_buf(v, "hb", (size_t)n * D * 4, &hb));
  TRY(vis_buf(v, "qkv", (size_t)n * 3 * D * 4, &qkv));
  TRY(vis_buf(v, "q", (size_t)n * kVisHeads * 304, &q));   // split rows of 304 bytes a head, or fp32 ones of 288
  TRY(vis_buf(v, "k", (size_t)n * kVisHeads * 304, &k));
  TRY(vis_buf(v, "vt", (size_t)np * D * 4, &vt));
  TRY(vis_buf(v, "att", (size_t)n * D * 4, &att));
  TRY(vis_buf(v, "up", (size_t)n * ((kVisF + 63) / 64 * 64) * 4, &up));
  const int most = std::max(vis_split(n, D, D), vis_split(n, D, (kVisF + 63) / 64 * 64));
  if (most > 1) TRY(vis_buf(v, "part", (size_t)most * n * D * 4, &part));
  HIPCHK(vis_prep(s, px, w, gh, gw, vis_t(v, "v.position_embd.weight"), v->side, D, pat, pe, cs));
  HIPCHK(vis_gemm(s, pat, v->pw, vis_t(v, "v.patch_embd.bias"), pe, x, n, D, 768, 0));
  float* tr = nullptr;
  if (v->trace) {
    TRY(vis_buf(v, "trace", (size_t)2 * n * D * 4, &tr));
    HIPCHK(hipMemcpyAsync(tr, x, (size_t)n * D * 4, hipMemcpyDeviceToDevice, s));
  }
  const float qscale = (float)(1.4426950408889634 / sqrt((double)kVisHd));
  int S = 0;                       // the parts that the residual stream still lacks
  const float* bias = nullptr;     // and their bias
  for (int i = 0; i <= kVisDepth; ++i) {
    // block i's first LayerNorm finishes block i - 1's rows, which the merger after i - 1 reads
    if (i < kVisDepth) {
      const VisBlock& b = v->blocks[i];
      TRY(vis_norm(v, n, D, x, S, part, bias, b.ln1w, b.ln1b, b.qkv, hb));
      S = 0;
    }
    if (i == 1 && tr) HIPCHK(hipMemcpyAsync(tr + (size_t)n * D, x, (size_t)n * D * 4, hipMemcpyDeviceToDevice, s));
    for (int j = 0; j < 3; ++j)
      if (kVisDeep[j] == i - 1) TRY(vis_merger(v, x, n, 0, nullptr, nullptr, deep + (size_t)j * m * kVisOut, j));
    if (i == kVisDepth) break;
    const VisBlock& b = v->blocks[i];
    TRY(vis_mm(v, b.qkv, hb, nullptr, qkv, n));
    if (b.heads) {
      HIPCHK(vis_heads_s(s, n, np, kVisHeads, qkv, cs, std::ldexp(qscale, b.eq), std::ldexp(1.f, b.ek),
                         std::ldexp(1.f, b.ev), (uint16_t*)q, (uint16_t*)k, (uint16_t*)vt));
      HIPCHK(vis_attend_s(s, n, np, kVisHeads, (const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)vt,
                          std::ldexp(1.f, -(b.eq + b.ek)), std::ldexp(1.f, -b.ev), D, b.out.split ? (uint16_t*)att : nullptr,
                          b.out.split ? nullptr : att));
    } else {
      HIPCHK(vis_heads(s, n, kVisHeads, qkv, cs, qscale, q, k, vt));
      HIPCHK(vis_attend(s, n, kVisHeads, q, k, vt, att));
    }
    TRY(vis_mm_add(v, b.out, att, x, n, S, part));
    TRY(vis_norm(v, n, D, x, S, part, b.out.b, b.ln2w, b.ln2b, b.up, hb));
    TRY(vis_mm_gelu(v, b.up, b.down, hb, up, n, 1));
    TRY(vis_mm_add(v, b.down, up, x, n, S, part));
    bias = b.down.b;
  }
  TRY(vis_merger(v, x, n, S, part, bias, merged, 3));
  if (tr) v->traced_n = n;
  return EXN_OK;
}


int exn_vision_encode_dev(exn_vision* v, const float* px, int h, int w, float* merged, float* deepstack) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  TRY(use(v->ctx));
  if (!px || !merged || !deepstack || h <= 0 || w <= 0 || h % 32 || w % 32 || (int64_t)(h / 16) * (w / 16) > 16384)
    FAIL(EXN_EINVAL, "vision encode: picture %d x %d (multiples of 32, at most 16384 patches)", h, w);
  TRY(exn_vision_check(v));
  return vis_encode(v, px, h, w, merged, deepstack);
}

int exn_vision_encode(exn_vision* v, const float* px, int h, int w, float* merged, float* deepstack) {
  if (!v) FAIL(EXN_EINVAL, "null vision tower");
  TRY(use(v->ctx));
  if (!px || !merged || !deepstack || h <= 0 || w <= 0 || h % 32 || w % 32 || (int64_t)(h / 16) * (w / 16) > 16384)
    FAIL(EXN_EINVAL, "vision encode: picture %d x %d (multiples of 32, at most 16384 patches)", h, w);
  const int64_t npx = (int64_t)h * w * 4, m = (int64_t)(h / 32) * (w / 32);
  float *dp, *dm;
  TRY(vis_buf(v, "h_px", (size_t)npx * 4, &dp));
  TRY(vis_buf(v, "h_out", (size_t)4 * m * kVisOut * 4, &dm));
  HIPCHK(hipMemcpyAsync(dp, px, (size_t)npx * 4, hipMemcpyHostToDevice, v->ctx->stream));
  TRY(exn_vision_encode_dev(v, dp, h, w, dm, dm + m * kVisOut));
  HIPCHK(hipMemcpyAsync(merged, dm, (size_t)m * kVisOut * 4, hipMemcpyDeviceToHost, v->ctx->stream));
  HIPCHK(hipMemcpyAsync(deepstack, dm + m * kVisOut, (size_t)3 * m * kVisOut * 4, hipMemcpyDeviceToHost,
                        v->ctx->stream));
  HIPCHK(hipStreamSynchronize(v->ctx->stream));
  return EXN_OK;
}

int exn_vision_traced(exn_vision* v, int which, float* out) {
  if (!v || !out || which < 0 || which > 1) FAIL(EXN_EINVAL, "vision traced: arguments");
  TRY(use(v->ctx));
  auto it = v->bufs.find("trace");
  if (!v->traced_n || it == v->bufs.end()) FAIL(EXN_ESTATE, "vision traced: no traced encode");
  const size_t rows = (size_t)v->traced_n * kVisD;
  HIPCHK(hipMemcpyAsync(out, (const float*)it->second.p + which * rows, rows * 4, hipMemcpyDeviceToHost,
                        v->ctx->stream));
  HIPCHK(hipStreamSynchronize(v->ctx->stream));
  return EXN_OK;
}

int exn_vis_gemm(exn_ctx* ctx, const float* x, const float* w, const float* bias, const float* r, float* y, int64_t m,
                 int64_t n, int64_t k, int act) {
  TRY(use(ctx));
  if (!x || !w || !bias || !y || act < 0 || act > 2) FAIL(EXN_EINVAL, "vis gemm arguments");
  const hipError_t e = vis_gemm(ctx->stream, x, w, bias, r, y, m, n, k, act);
  if (e == hipErrorInvalidValue) FAIL(EXN_EINVAL, "vis gemm: %lld x %lld x %lld", (long long)m, (long long)n, (long long)k);
  HIPCHK(e);
  return EXN_OK;
}

int exn_vis_attend(exn_ctx* ctx, int n, int heads, const float* q, const float* k, const float* vt, float* att) {
  TRY(use(ctx));
  if (!q || !k || !vt || !att || n <= 0 || heads <= 0) FAIL(EXN_EINVAL, "vis attend arguments");
  const hipError_t e = vis_attend(ctx->stream, n, heads, q, k, vt, att);
  if (e == hipErrorInvalidValue) FAIL(EXN_EINVAL, "vis attend: n %d (a multiple of 4)", n);
  HIPCHK(e);
  return EXN_OK;
}

int exn_vis_ln(exn_ctx* ctx, int64_t rows, int width, const float* x, const float* w, const float* b, float* y) {
  TRY(use(ctx));
  if (!x || !w || !b || !y || rows < 0) FAIL(EXN_EINVAL, "vis ln arguments");
  const hipError_t e = vis_ln_s(ctx->stream, rows, width, 0, (float*)x, 0, nullptr, nullptr, w, b, 1.f, nullptr, y);
  if (e == hipErrorInvalidValue) FAIL(EXN_EINVAL, "vis ln: width %d (a multiple of 4, at most 5120)", width);
  HIPCHK(e);
  return EXN_OK;
}

int exn_vis_gemm_way(int64_t m, int64_t n, int64_t kp, int parts, int* tile, int* pays) {
  if (!tile || !pays || m <= 0 || n <= 0 || kp < 64 || kp % 64 || parts < 1 || parts > kp / 64)
    FAIL(EXN_EINVAL, "vis gemm way arguments");
  *tile = vis_tile(m, n, kp, parts);
  *pays = vis_split(m, n, kp);
  return EXN_OK;
}

int exn_vis_gemm_s(exn_ctx* ctx, const uint16_t* x, const uint16_t* w, const float* bias, const float* r, float* y,
                   uint16_t* ys, int64_t m, int64_t n, int64_t kp, float descale, float oscale, int64_t ldy, int act,
                   int parts) {
  TRY(use(ctx));
  if (!x || !w || !y == !ys || parts < 1 || (parts > 1 ? !y || r || act : !bias)) FAIL(EXN_EINVAL, "vis gemm_s arguments");
  const hipError_t e = parts > 1 ? vis_gemm_part(ctx->stream, x, w, y, m, n, kp, descale, parts)
                                 : vis_gemm_s(ctx->stream, x, w, bias, r, y, ys, m, n, kp, descale, oscale, ldy, act);
  if (e == hipErrorInvalidValue)
    FAIL(EXN_EINVAL, "vis gemm_s: %lld x %lld x %lld, %d parts", (long long)m, (long long)n, (long long)kp, parts);
  HIPCHK(e);
  return EXN_OK;
}

int exn_vis_ln_s(exn_ctx* ctx, int64_t rows, int width, float* x, int parts, const float* part, const float* bias,
                 const float* w, const float* b, float scale, uint16_t* ys, float* yf) {
  TRY(use(ctx));
  if (!x || !w || !b || rows < 0 || (parts > 0 && (!part || !bias))) FAIL(EXN_EINVAL, "vis ln_s arguments");
  const hipError_t e = vis_ln_s(ctx->stream, rows, width, width, x, parts, part, bias, w, b, scale, ys, yf);
  if (e == hipErrorInvalidValue) FAIL(EXN_EINVAL, "vis ln_s: width %d (a multiple of 64, at most 5120)", width);
  HIPCHK(e);
  return EXN_OK;
}

int exn_vis_heads_s(exn_ctx* ctx, int n, int heads, const float* qkv, const float* cs, float qs, float ks, float vs,
                    uint16_t* q, uint16_t* k, uint16_t* vt) {
  TRY(use(ctx));
  if (!qkv || !cs || !q || !k || !vt || n <= 0 || heads <= 0) FAIL(EXN_EINVAL, "vis heads_s arguments");
  HIPCHK(vis_heads_s(ctx->stream, n, (n + 63) / 64 * 64, heads, qkv, cs, qs, ks, vs, q, k, vt));
  return EXN_OK;
}

int exn_vis_attend_s(exn_ctx* ctx, int n, int heads, const uint16_t* q, const uint16_t* k, const uint16_t* vt, float sc,
                     float vde, uint16_t* ys, float* yf) {
  TRY(use(ctx));
  if (!q || !k || !vt || !ys == !yf || n <= 0 || heads <= 0 || (ys && heads * 72 % 64))
    FAIL(EXN_EINVAL, "vis attend_s arguments");
  HIPCHK(vis_attend_s(ctx->stream, n, (n + 63) / 64 * 64, heads, q, k, vt, sc, vde, heads * 72, ys, yf));
  return EXN_OK;
}

int exn_vis_spread(exn_ctx* ctx, int rows, int cols, const float* w, const float* g, const float* b, int period,
                   const float* bias, int gelu, double* a2, double* t2, double* spread2) {
  TRY(use(ctx));
  if (!w || !g || !b || !bias || !a2 || !t2 || !spread2 || rows <= 0 || cols <= 0 || cols % 4 || period <= 0 || period % 4)
    FAIL(EXN_EINVAL, "vis spread arguments");
  HIPCHK(tensor_stats_clear(ctx->stream, (uint32_t*)spread2, 1));
  HIPCHK(vis_square(ctx->stream, period, g, b, a2));
  HIPCHK(vis_rows(ctx->stream, rows, cols, w, a2, period, bias, gelu, t2, spread2));
  return EXN_OK;
}
