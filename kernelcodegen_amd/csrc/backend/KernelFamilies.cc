#include "backend/KernelFamilies.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <sstream>
#include <vector>

// Generated at build time from backend/kernels/*.hip: one raw string per file.
#include "backend/kernels/_templates_gen.inc"

namespace KernelCodeGen {
namespace hipgen {

namespace {

struct Defines {
  std::vector<std::pair<std::string, std::string>> items;
  void add(const std::string& k, const std::string& v) { items.emplace_back(k, v); }
  void add(const std::string& k, int64_t v) { items.emplace_back(k, std::to_string(v)); }
  std::string wrap(const char* body) const {
    std::ostringstream os;
    for (auto& kv : items) os << "#define " << kv.first << " " << kv.second << "\n";
    os << body << "\n";
    for (auto& kv : items) os << "#undef " << kv.first << "\n";
    return os.str();
  }
};

std::string floatLiteral(double v) {
  char buf[64];
  snprintf(buf, sizeof buf, "%af", (double)(float)v);  // hex float: exact fp32 value
  return buf;
}

int64_t ceilDiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

int64_t nextPow2(int64_t v) {
  int64_t p = 1;
  while (p < v) p <<= 1;
  return p;
}

bool need(const KernelSpec& s, std::initializer_list<const char*> keys, std::string& err) {
  for (auto k : keys)
    if (!s.has(k)) {
      err = "kernel family '" + s.family + "' needs parameter " + k;
      return false;
    }
  return true;
}

bool positive(const KernelSpec& s, std::initializer_list<const char*> keys, std::string& err) {
  for (auto k : keys)
    if (s.get(k, 0) <= 0) {
      err = std::string("parameter ") + k + " must be positive";
      return false;
    }
  return true;
}

// ---------------------------------------------------------------------------
bool emitLayerNorm(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  if (!need(s, {"ROWS", "N"}, err) || !positive(s, {"ROWS", "N"}, err)) return false;
  const int64_t rows = s.p["ROWS"], n = s.p["N"];
  const int64_t ng = s.get("NG", n), nb = s.get("NB", n);
  if (ng <= 0 || nb <= 0 || n % ng || n % nb) {
    err = "layernorm: scale/bias length must divide the normalised length";
    return false;
  }
  const bool f16 = s.get("F16", 0) != 0;
  const double elements = (double)rows * (double)n;
  auto divides = [&](int64_t w) { return n % w == 0 && ng % w == 0 && nb % w == 0; };
  // Rows of 512 to 8192 elements, for callers who ask for it (FILL = 2) and on more than 1024 rows: 16 bytes per access whatever the
  // length, and the fewest lanes that hold a row in `most` vectors each, since a lane past the row's end idles as long as the others
  // work (bf16, 640 vectors a row: 128 lanes of five against 512 of which 320 take two).  Up to 256 rows the launch is one row's chain,
  // which more lanes shorten; up to 2048 the part is not full yet.  Scale and bias are then read again by every row (they come out of
  // the caches) and rows have a workgroup each, without a next row under way: more wavefronts fit a CU that way than the held
  // values' registers leave.  Where rows fill the registers all the same, and in fp32, large launches stay with 512 workgroups that
  // hold and prefetch.  us, before and now, bf16: 16384 x 5120 89 and 58, 4000 x 2560 12.7 and 6.6, 1100 x 6144 10.4 and 5.1, 100 x 1280
  // 3.15 and 2.43, 16384 x 4096 49.7 and 45.8, odd lengths 16384 x 1001 31.7 and 14.2, 4000 x 2503 21.8 and 8.5, 16384 x 7777 138 and 106;
  // fp32 16384 x 1280 34.7 and 28.6, 1100 x 4096 8.4 and 6.3, 16384 x 3333 81 and 74.  Held and prefetched, and neither: bf16 16384 x 8192
  // 86 and 95, 4000 x 7777 28.8 and 30.4, but 4000 x 7168 24.1 and 22.9; fp32 4000 x 2560 15.8 and 16.9, but 4000 x 1280 7.5 and 6.7,
  // 16384 x 640 17.0 and 15.7 (but 9208 x 948 13.0 and 14.9).
  const int64_t wide = f16 ? 8 : 4;
  bool tuned = (s.get("FILL", 0) >= 2 || rows > 1024) && n >= 512 && n <= 8192 && ((ng == n && nb == n) || divides(wide));
  for (const char* key : {"VW", "TPR", "RPB", "GRID", "LEAN", "ONEPASS"}) tuned = tuned && !s.has(key);
  if (tuned) {
    const bool hold = rows <= 256 || (f16 ? n > 6144 && elements > 24e6 : n > 768 && elements > (n <= 1024 ? 6e6 : 8e6));
    // (fp32: a wavefront by itself up to 1024, 1 x 576 2.03 us and 2.11; held rows beyond 4096 on 512 lanes, 16384 x 5120 111 and 114)
    const int64_t most = f16 ? (rows <= 256 ? 1 : rows <= 2048 ? 3 : 6) : rows > 256 ? 5 : n > 1024 ? 1 : 4;
    int64_t lanes = 64;
    while (lanes * most * wide < n && lanes < 256) lanes *= 2;
    if (lanes * 6 * wide < n || (!f16 && rows > 256 && hold && n > 4096)) lanes = 512;
    s.p["VW"] = wide; s.p["TPR"] = lanes;
    s.p["LEAN"] = !hold;
    // Held rows walk on 512 workgroups, up to 1024 elements on 768 (fp32 16384 x 832 19.5 us and 21.0, 9208 x 948 13.0 and 13.6), and so do
    // fp32 rows that start off the vectors on teams of 128 and 256 while they are not many more than the caches hold: 512 and 768, 4926 x
    // 2639 23.3 and 19.4, 8684 x 1497 21.3 and 19.7, 3241 x 4010 20.0 and 18.5; but 16004 x 3999 85 and 90.
    const bool off = !f16 && n % wide != 0 && lanes >= 128 && lanes <= 256 && elements <= 32e6;
    s.p["GRID"] = hold && rows > 256 ? (n <= 1024 || off ? 768 : 512) : rows;
  }
  // Else 16 bytes per access where all lengths divide into them (16-bit types fall back to fours), and on launches of at least a
  // million elements of any row length, scale and bias then being of that length; smaller odd launches and short rows, where most of
  // a wavefront would idle, keep single elements, and so do 16-bit rows of 2048 to 4096 while every row has a workgroup to itself
  // (512), and those where the eights take too many registers (beyond 8192; fp32 in fours stays ahead to the 32 elements a lane holds):
  // bf16 us, eights and single elements, 2100 x 16381 53 and 42, but 1000 x 8191 9.8 and 12.8.
  // 16-bit rows that fours divide and eights do not go in fours, aligned as they are, while those leave a lane half a vector free
  // (7168), on up to 4096 elements by 1024 workgroups.
  const bool anyLength = ng == n && nb == n && n >= 256 && n <= (f16 ? 8192 : 1024 * 32) && elements >= 1048576.0 &&
                         !(f16 && n > 2048 && n <= 4096 && rows <= 512);
  // (a wavefront that fours fill and eights do not, 768 elements: fours on small launches, 300 x 768 3.2 us and 3.0)
  const bool unfilled = f16 && n < 1024 && n % 256 == 0 && n % 512 != 0 && elements <= 2097152.0;
  const bool fours = divides(4) && f16 && n >= 1024 && n <= 7168;
  int64_t vw = s.get("VW", divides(wide) && n >= 512 && !unfilled ? wide : anyLength && !fours ? (n >= 1024 ? wide : 4) : divides(4) ? 4 : 1);
  if (vw != 1 && vw != 4 && vw != 8) { err = "layernorm: VW must be 1, 4 or 8"; return false; }
  if (vw > 1 && s.has("VW") && !tuned && !divides(vw)) { err = "layernorm: VW=" + std::to_string(vw) + " needs lengths divisible by " + std::to_string(vw); return false; }
  int64_t tpr = s.get("TPR", 0);
  if (rows > 0xFFFFFFFFLL) { err = "layernorm: too many rows"; return false; }
  if (tpr == 0) {
    // Four vectors per lane measured best for 4096-float rows, with and without the GELU; of 16-bit values, eight to a vector,
    // two (so as many lanes as with fours: half of them made small launches slower than fours, bf16 us with four vectors, two,
    // and in fours: 1 x 4096 3.24, 2.76, 3.11; 64 x 2048 3.44, 2.89, 3.34; 4000 x 4096 17.9, 14.7, 18.7; 16384 x 4096 68, 50, 66; 12000 x 3333 66, 55),
    // but three where one wavefront then holds the row (64 x 1536 3.14 us, 3.33 on two).
    tpr = nextPow2(ceilDiv(n, vw * (vw == 8 && n > 1536 ? 2 : 4)));
    if (tpr < 64) tpr = 64;
    if (tpr > 512) tpr = 512;
  }
  if (tpr < 64 || tpr > 1024 || (tpr & (tpr - 1))) { err = "layernorm: TPR must be a power of two in [64,1024]"; return false; }
  int64_t vpt = ceilDiv(n, tpr * vw);
  const int64_t few = vw == 8 ? 4 : 8;     // vectors per lane that leave room for gamma, beta and a second row in registers
  if (vpt > few && !s.has("TPR")) {  // widen the team: up to 8 vectors per lane leave room for gamma, beta and a prefetched row
    tpr = 1024;
    vpt = ceilDiv(n, tpr * vw);
  }
  const double esize = f16 ? 2.0 : 4.0;
  if (vpt > (vw == 8 ? 16 : 32)) {
    // the group does not fit the register file of one workgroup: three streamed passes
    const int64_t block = 1024;
    if (!divides(vw)) vw = divides(4) ? 4 : 1;
    s.p["VW"] = vw; s.p["TPR"] = block; s.p["RPB"] = 1; s.p["VPT"] = 0; s.p["NG"] = ng; s.p["NB"] = nb;
    Defines d;
    d.add("LS_NAME", s.name);
    d.add("LS_ROWS", rows);
    d.add("LS_N", std::to_string(n) + "L");
    d.add("LS_NG", ng);
    d.add("LS_NB", nb);
    d.add("LS_EPS", floatLiteral(s.f.count("EPS") ? s.f["EPS"] : 1e-5));
    d.add("LS_BLOCK", block);
    d.add("LS_VW", vw);
    d.add("LS_GELU", s.get("GELU", 0) ? 1 : 0);
    d.add("LS_F16", s.get("F16", 0));
    src = d.wrap(kTpl_layernorm_stream);
    info.name = s.name;
    info.grid[0] = (uint32_t)rows;
    info.block[0] = (uint32_t)block;
    info.numArgs = 4;
    info.flops = 8.0 * (double)rows * (double)n;
    info.bytes = 2.0 * (double)rows * (double)n * esize + (double)(ng + nb) * esize;
    return true;
  }
  int64_t rpb = s.get("RPB", tpr >= 256 ? 1 : 256 / tpr);
  if (rpb < 1 || rpb * tpr > 1024) { err = "layernorm: RPB*TPR must be in [64,1024]"; return false; }
  s.p["VW"] = vw; s.p["TPR"] = tpr; s.p["RPB"] = rpb; s.p["VPT"] = vpt; s.p["NG"] = ng; s.p["NB"] = nb;

  Defines d;
  d.add("LN_NAME", s.name);
  d.add("LN_ROWS", rows);
  d.add("LN_N", n);
  d.add("LN_NG", ng);
  d.add("LN_NB", nb);
  d.add("LN_EPS", floatLiteral(s.f.count("EPS") ? s.f["EPS"] : 1e-5));
  d.add("LN_TPR", tpr);
  d.add("LN_RPB", rpb);
  d.add("LN_VW", vw);
  d.add("LN_VPT", vpt);
  d.add("LN_GELU", s.get("GELU", 0) ? 1 : 0);
  d.add("LN_F16", s.get("F16", 0));
  // Two persistent workgroups per CU, each walking the row groups with stride GRID and loading its next
  // row before it reduces the current one: measured on operands that are not in the last-level cache
  // (three rotating buffer sets), 16384 x 4096 runs at 6.1 TB/s this way against 5.5 TB/s with one
  // workgroup per row; a plain copy reaches 6.3-6.4 TB/s under the same conditions.
  const int64_t groups = ceilDiv(rows, rpb);
  int64_t grid = s.get("GRID", 0);
  // (four per CU where a lane's share of a row is two vectors of eight: bf16 16384 x 1000 13.3 us against 16.9; or four of
  // four: 16384 x 3892 66 against 85)
  // A lane of 1024, which has 128 registers, has no room for gamma, beta and a second row beside more than 24 values of its row
  // either: 88-212 bytes of scratch (bf16 2000 x 25600 87 us, 44 without the prefetch; fp32 1000 x 28135 70 and 47)
  const bool crowded = vpt > few || (tpr == 1024 && vpt * vw > 24);
  const bool wideGrid = f16 && ((vw == 8 && vpt <= 2) || (vw == 4 && n >= 1024 && n <= 4096));
  if (grid <= 0) grid = crowded ? groups : wideGrid ? 1024 : 512;      // rows too long to prefetch keep one workgroup per group
  // (a launch takes fewer than 2^32 threads: 2^26 rows of 512, a wavefront each, are one workgroup too many; the rest is walked)
  grid = std::min({grid, groups, (int64_t)(0xFFFFFFFFLL / (tpr * rpb))});
  s.p["GRID"] = grid;
  d.add("LN_GRID", grid);
  d.add("LN_STREAM", s.get("STREAM", 1) ? 1 : 0);
  d.add("LN_LEAN", s.get("LEAN", crowded ? 1 : 0) ? 1 : 0);
  // one reduction per row (merged means and sums of squared deviations) where every lane holds the same number of values
  const bool onePass = s.get("ONEPASS", 0) != 0 && n % (tpr * vw) == 0;
  s.p["ONEPASS"] = onePass;
  d.add("LN_ONEPASS", onePass ? 1 : 0);
  src = d.wrap(kTpl_layernorm);

  info.name = s.name;
  info.grid[0] = (uint32_t)grid;
  info.block[0] = (uint32_t)(tpr * rpb);
  info.numArgs = 4;
  info.flops = 8.0 * (double)rows * (double)n;
  info.bytes = 2.0 * (double)rows * (double)n * esize + (double)(ng + nb) * esize;
  return true;
}

// ---------------------------------------------------------------------------
bool parseList(const std::string& text, std::vector<int64_t>& out) {
  out.clear();
  std::stringstream ss(text);
  std::string item;
  while (std::getline(ss, item, ',')) {
    if (item.empty()) return false;
    char* end = nullptr;
    const long long v = std::strtoll(item.c_str(), &end, 10);
    if (*end) return false;
    out.push_back(v);
  }
  return !out.empty();
}

std::string joinList(const std::vector<int64_t>& v) {
  std::string s;
  for (size_t i = 0; i < v.size(); ++i) s += (i ? ", " : "") + std::to_string(v[i]) + "L";
  return s;
}

bool emitBinary(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  static const char* names[] = {"Add", "Sub", "Mul", "Div", "Pow", "Equal", "Greater"};
  int op = -1;
  for (int i = 0; i < 7; ++i)
    if (s.s.count("OP") && s.s["OP"] == names[i]) op = i;
  if (op < 0) { err = "binary: OP must be Add, Sub, Mul, Div, Pow, Equal or Greater"; return false; }
  const bool compare = op >= 5;     // one byte per result element
  std::vector<int64_t> dims, sa, sb;
  if (!s.s.count("DIMS") || !s.s.count("SA") || !s.s.count("SB") || !parseList(s.s["DIMS"], dims) ||
      !parseList(s.s["SA"], sa) || !parseList(s.s["SB"], sb) || sa.size() != dims.size() || sb.size() != dims.size()) {
    err = "binary: DIMS, SA and SB must be comma separated lists of one length";
    return false;
  }
  if (dims.size() > 6) { err = "binary: rank above 6"; return false; }
  int64_t total = 1, elemsA = 1, elemsB = 1;
  for (size_t d = 0; d < dims.size(); ++d) {
    if (dims[d] <= 0 || sa[d] < 0 || sb[d] < 0) { err = "binary: extents must be positive and strides non-negative"; return false; }
    total *= dims[d];
    if (sa[d]) elemsA *= dims[d];
    if (sb[d]) elemsB *= dims[d];
  }
  const bool inplace = s.get("INPLACE", 0) != 0;
  if (inplace && elemsA != total) { err = "binary: an in-place result needs an unbroadcast left operand"; return false; }
  if (inplace && compare) { err = "binary: a comparison cannot overwrite its fp32 operand"; return false; }
  const int64_t inner = dims.back();
  const bool lastOk = (sa.back() == 1 || sa.back() == 0) && (sb.back() == 1 || sb.back() == 0);
  if (!lastOk) { err = "binary: the innermost stride of an operand must be 1 or 0"; return false; }
  // 128-bit accesses need every operand row to start on a 16-byte boundary
  bool aligned = inner % 4 == 0;
  for (size_t d = 0; d + 1 < dims.size(); ++d) aligned = aligned && sa[d] % 4 == 0 && sb[d] % 4 == 0;
  int64_t vw = s.get("VW", aligned ? 4 : 1);
  if (vw != 1 && vw != 4) { err = "binary: VW must be 1 or 4"; return false; }
  if (vw == 4 && !aligned) { err = "binary: VW=4 needs rows that are multiples of four elements"; return false; }
  int64_t block = s.get("BLOCK", 512);
  if (block < 64 || block > 1024 || block % 64) { err = "binary: bad BLOCK"; return false; }
  if (ceilDiv(total, vw * block) > 0x7FFFFFFFLL) { err = "binary: too many elements"; return false; }
  s.p["VW"] = vw; s.p["BLOCK"] = block;

  Defines d;
  d.add("BN_NAME", s.name);
  d.add("BN_RANK", (int64_t)dims.size());
  d.add("BN_DIMS", joinList(dims));
  d.add("BN_SA", joinList(sa));
  d.add("BN_SB", joinList(sb));
  d.add("BN_OP", op);
  d.add("BN_VW", vw);
  d.add("BN_BLOCK", block);
  d.add("BN_INPLACE", inplace ? 1 : 0);
  d.add("BN_F16", s.get("F16", 0) ? 1 : 0);
  // An operand that is not broadcast is read once: non-temporal loads for it (bit 0: X, bit 1: Y); a broadcast one is
  // read again and again out of the cache and keeps plain loads (16384 x 4096 plus a row: 84.3 us with the hint on X
  // alone, 86.0 without, 86.5 with it on both).  Not for an in-place result, whose operand is written back.
  const int64_t stream = s.get("STREAM", inplace ? 0 : ((elemsA == total ? 1 : 0) | (elemsB == total ? 2 : 0))) & 3;
  s.p["STREAM"] = stream;
  d.add("BN_STREAM", stream);
  src = d.wrap(kTpl_binary);

  info.name = s.name;
  info.grid[0] = (uint32_t)ceilDiv(total, vw * block);
  info.block[0] = (uint32_t)block;
  info.numArgs = inplace ? 2 : 3;
  info.flops = (double)total;
  const double esize = s.get("F16", 0) ? 2.0 : 4.0;
  info.bytes = esize * ((double)elemsA + (double)elemsB) + (compare ? 1.0 : esize) * (double)total;
  return true;
}

bool emitSoftmax(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  if (!need(s, {"ROWS", "N"}, err) || !positive(s, {"ROWS", "N"}, err)) return false;
  const int64_t rows = s.p["ROWS"], n = s.p["N"];
  // As for LayerNorm: 16 bytes per access where the length divides into them, and on large launches of any length (us, single
  // elements, fours, 16 bytes: bf16 12000 x 2048 41.7, 18.7, 16.5; 4096 x 4096 29.9, 13.5, 9.6; 2000 x 32000 138, 68, 47;
  // 12000 x 2047 42.9, 22.6, 20.6; 30000 x 257 20.3, 12.1, 14.6; 100 x 1001 3.3, 3.9).  16-bit rows
  // that fours divide and eights do not go in fours on launches of up to 8 M elements (eights with a ragged end and fours: 300 x
  // 3892 4.7 and 4.0, 1000 x 8188 7.7 and 7.2); on larger ones eights are ahead or within 6 % (4000 x 3892 12.2 and 13.9, 8000 x 2044
  // 13.2 and 13.9, 16384 x 1500 22.3 and 21.3, 16384 x 3892 51.8 and 48.9).
  const bool f16 = s.get("F16", 0) != 0;
  const int64_t wide = f16 ? 8 : 4;
  const double elements = (double)rows * (double)n;
  const bool small = elements <= 4194304.0;
  const bool anyLength = n >= 256 && n <= 1024 * 32 && elements >= 1048576.0;
  const bool fours = n % 4 == 0 && f16 && n >= 1024 && elements <= 8388608.0;
  int64_t vw = s.get("VW", n % wide == 0 && n >= 512 ? wide : anyLength && !fours ? (n >= 1024 ? wide : 4) : n % 4 == 0 ? 4 : 1);
  if (vw != 1 && vw != 4 && vw != 8) { err = "softmax: VW must be 1, 4 or 8"; return false; }
  if (vw > 1 && s.has("VW") && n % vw) { err = "softmax: VW=" + std::to_string(vw) + " needs a row length divisible by " + std::to_string(vw); return false; }
  int64_t tpr = s.get("TPR", 0);
  if (tpr == 0) {
    // About four vectors per lane; on small launches two of eights, as many lanes as fours have (bf16 us with four vectors,
    // two, and in fours: 1 x 4096 3.09, 2.65, 2.91; 300 x 2048 3.35, 2.99, 3.22; 1000 x 4096 5.2, 4.35, 4.5; 1000 x 3893 7.2, 6.5; but 4000 x 4096 10.6, 12.5)
    tpr = nextPow2(ceilDiv(n, vw * (vw == 8 && n > 1536 && n <= (n % 8 ? 4096 : 8192) && small ? 2 : 4)));
    if (tpr < 64) tpr = 64;
    if (tpr > 1024) tpr = 1024;
  }
  if (tpr < 64 || tpr > 1024 || (tpr & (tpr - 1))) { err = "softmax: TPR must be a power of two in [64,1024]"; return false; }
  const int64_t vpt = ceilDiv(n, tpr * vw);
  if (vpt > (vw == 8 ? 16 : 32)) {
    if (n % vw) vw = n % 4 == 0 ? 4 : 1;
    // rows too long for registers (a vocabulary of 150 000 logits, say): one workgroup per row, two streamed passes
    if (rows > 0x7FFFFFFFLL) { err = "softmax: too many rows"; return false; }
    const bool inplaceLong = s.get("INPLACE", 1) != 0;
    s.p["VW"] = vw; s.p["TPR"] = 1024; s.p["RPB"] = 1; s.p["VPT"] = 0; s.p["INPLACE"] = inplaceLong;
    Defines d;
    d.add("SS_NAME", s.name);
    d.add("SS_ROWS", rows); d.add("SS_N", n);
    d.add("SS_BLOCK", 1024); d.add("SS_VW", vw);
    d.add("SS_INPLACE", inplaceLong ? 1 : 0);
    d.add("SS_F16", s.get("F16", 0));
    src = d.wrap(kTpl_softmax_stream);
    info.name = s.name;
    info.grid[0] = (uint32_t)rows;
    info.block[0] = 1024;
    info.numArgs = inplaceLong ? 1 : 2;
    info.flops = 4.0 * (double)rows * (double)n;
    info.bytes = 2.0 * (double)rows * (double)n * (s.get("F16", 0) ? 2.0 : 4.0);
    return true;
  }
  int64_t rpb = s.get("RPB", tpr >= 256 ? 1 : 256 / tpr);
  if (rpb < 1 || rpb * tpr > 1024) { err = "softmax: RPB*TPR must be in [64,1024]"; return false; }
  const int64_t groups = ceilDiv(rows, rpb);
  if (groups > 0x7FFFFFFFLL) { err = "softmax: too many rows"; return false; }
  const bool inplace = s.get("INPLACE", 1) != 0;
  s.p["VW"] = vw; s.p["TPR"] = tpr; s.p["RPB"] = rpb; s.p["VPT"] = vpt; s.p["INPLACE"] = inplace;

  Defines d;
  d.add("SM_NAME", s.name);
  d.add("SM_ROWS", rows); d.add("SM_N", n);
  d.add("SM_TPR", tpr); d.add("SM_RPB", rpb); d.add("SM_VW", vw); d.add("SM_VPT", vpt);
  d.add("SM_INPLACE", inplace ? 1 : 0);
  d.add("SM_STREAM", s.get("STREAM", 1) ? 1 : 0);
  d.add("SM_F16", s.get("F16", 0));
  src = d.wrap(kTpl_softmax);

  info.name = s.name;
  info.grid[0] = (uint32_t)groups;
  info.block[0] = (uint32_t)(tpr * rpb);
  info.numArgs = inplace ? 1 : 2;
  info.flops = 4.0 * (double)rows * (double)n;
  info.bytes = 2.0 * (double)rows * (double)n * (s.get("F16", 0) ? 2.0 : 4.0);
  return true;
}

bool emitGather(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  if (!need(s, {"OUTER", "AXIS", "NIDX", "INNER", "ESIZE"}, err) || !positive(s, {"OUTER", "AXIS", "NIDX", "INNER", "ESIZE"}, err))
    return false;
  const int64_t outer = s.p["OUTER"], axis = s.p["AXIS"], nidx = s.p["NIDX"], inner = s.p["INNER"], esize = s.p["ESIZE"];
  if (esize != 1 && esize != 2 && esize != 4 && esize != 8) { err = "gather: ESIZE must be 1, 2, 4 or 8 bytes"; return false; }
  const int64_t row = inner * esize;
  int64_t vb = 16;
  while (vb > 2 && row % vb) vb /= 2;
  if (row % vb) { err = "gather: rows of an odd number of bytes are not supported"; return false; }
  const int64_t block = s.get("BLOCK", 256);
  if (block < 64 || block > 1024 || block % 64) { err = "gather: bad BLOCK"; return false; }
  const double units = (double)outer * (double)nidx * (double)(row / vb);
  if (units / (double)block > 2147483647.0) { err = "gather: too many elements"; return false; }
  // two units per lane when there is work for every CU several times over (32000 x 4096 bf16 table, 16384 rows
  // picked, operands in HBM: 0.82 of the HBM peak against 0.78 with one unit, 0.75 with four)
  const int64_t unroll = s.get("UNROLL", units >= 2.0 * (double)block * 2048.0 ? 2 : 1);
  if (unroll < 1 || unroll > 16) { err = "gather: UNROLL must be in [1,16]"; return false; }
  s.p["BLOCK"] = block; s.p["VB"] = vb; s.p["UNROLL"] = unroll;

  Defines d;
  d.add("GA_NAME", s.name);
  d.add("GA_OUTER", outer); d.add("GA_AXIS", axis); d.add("GA_NIDX", nidx);
  d.add("GA_ROW", row); d.add("GA_VB", vb); d.add("GA_BLOCK", block); d.add("GA_UNROLL", unroll);
  src = d.wrap(kTpl_gather);

  info.name = s.name;
  info.grid[0] = (uint32_t)ceilDiv(outer * nidx * (row / vb), block * unroll);
  info.block[0] = (uint32_t)block;
  info.numArgs = 3;
  info.flops = 0.0;
  info.bytes = 2.0 * (double)outer * (double)nidx * (double)row + 8.0 * (double)nidx;   // rows read and written, indices
  return true;
}

// ---------------------------------------------------------------------------
int elementwiseOpCode(const std::string& op) {
  static const char* names[] = {"Tanh", "Sqrt", "Log", "Relu", "Gelu", "Cast"};
  for (int i = 0; i < 6; ++i)
    if (op == names[i]) return i;
  return -1;
}

int ctypeSize(const std::string& t) {
  if (t == "float" || t == "int") return 4;
  if (t == "double" || t == "long") return 8;
  if (t == "short" || t == "_Float16" || t == "__bf16") return 2;
  return 0;
}

bool emitElementwise(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  if (!need(s, {"N"}, err) || !positive(s, {"N"}, err)) return false;
  const int64_t n = s.p["N"];
  int op = s.has("OP") ? (int)s.p["OP"] : elementwiseOpCode(s.s.count("OP") ? s.s["OP"] : "");
  if (op < 0 || op > 5) { err = "elementwise: unknown operation"; return false; }
  std::string inT = s.s.count("IN_T") ? s.s["IN_T"] : "float";
  std::string outT = s.s.count("OUT_T") ? s.s["OUT_T"] : "float";
  if (!ctypeSize(inT) || !ctypeSize(outT)) { err = "elementwise: unsupported element type"; return false; }
  // the maps compute in fp32; operands and results are fp32, IEEE half or bfloat16 (converted on the way in and out)
  const bool floatIO = (inT == "float" || inT == "_Float16" || inT == "__bf16") && inT == outT;
  if (op != 5 && !floatIO) { err = "elementwise: only Cast changes the element type; the other maps take float, _Float16 or __bf16"; return false; }
  const bool inplace = s.get("INPLACE", 0) != 0;
  if (inplace && ctypeSize(inT) != ctypeSize(outT)) { err = "elementwise: in-place needs equal element sizes"; return false; }
  int64_t vw = s.get("VW", n % 4 == 0 ? 4 : 1);
  if (vw != 1 && vw != 4) { err = "elementwise: VW must be 1 or 4"; return false; }
  if (vw == 4 && n % 4) { err = "elementwise: VW=4 needs N divisible by 4"; return false; }
  int64_t block = s.get("BLOCK", 512), unroll = s.get("UNROLL", 1);
  if (block < 64 || block > 1024 || block % 64 || unroll < 1 || unroll > 16) { err = "elementwise: bad BLOCK/UNROLL"; return false; }
  s.p["VW"] = vw; s.p["BLOCK"] = block; s.p["UNROLL"] = unroll; s.p["OP"] = op;

  Defines d;
  d.add("EW_NAME", s.name);
  d.add("EW_N", std::to_string(n) + "L");
  d.add("EW_OP", op);
  d.add("EW_VW", vw);
  d.add("EW_BLOCK", block);
  d.add("EW_UNROLL", unroll);
  d.add("EW_STREAM", s.get("STREAM", 1) ? 1 : 0);
  d.add("EW_INPLACE", inplace ? 1 : 0);
  d.add("EW_IN_T", inT);
  d.add("EW_OUT_T", outT);
  src = d.wrap(kTpl_elementwise);

  info.name = s.name;
  info.grid[0] = (uint32_t)ceilDiv(n, vw * block * unroll);
  info.block[0] = (uint32_t)block;
  info.numArgs = inplace ? 1 : 2;
  info.flops = (op == 4 ? 10.0 : 1.0) * (double)n;
  info.bytes = (double)n * (ctypeSize(inT) + ctypeSize(outT));
  return true;
}

// ---------------------------------------------------------------------------
bool gemmCommon(KernelSpec& s, std::string& err, int64_t& m, int64_t& n, int64_t& k, int64_t& batch) {
  if (!need(s, {"M", "N", "K"}, err) || !positive(s, {"M", "N", "K"}, err)) return false;
  m = s.p["M"]; n = s.p["N"]; k = s.p["K"];
  batch = s.get("BATCH", 1);
  if (batch < 1 || batch > 65535) { err = "gemm: BATCH must be in [1,65535]"; return false; }
  if (m > (1LL << 30) || n > (1LL << 30) || k > (1LL << 30)) { err = "gemm: dimension too large"; return false; }
  return true;
}

bool checkTile(const KernelSpec& s, int64_t bm, int64_t bn, int64_t bk, int64_t wm, int64_t wn, int64_t kmul,
               std::string& err) {
  if (wm < 1 || wn < 1 || wm * wn > 16 || bm % (32 * wm) || bn % (32 * wn) || bk % kmul || bm <= 0 || bn <= 0 ||
      bk <= 0) {
    err = s.family + ": tile BM/BN must be multiples of 32*WM / 32*WN and BK a multiple of " + std::to_string(kmul);
    return false;
  }
  return true;
}

// Rows short enough that a lane's offset within the rows of one direct load (at most 64 rows where rows are clamped) stays
// in 32 bits: where more than the whole tiles of the direct-load kernels is taken, longer ones keep the other kernels.
static bool shortRows(int64_t n, int64_t k) { return n <= (1 << 23) && k <= (1 << 23); }

// Whether a caller names nothing but the problem: a kernel that has no use for some other wish is not taken in its place.
static bool namesOnly(const KernelSpec& s, std::initializer_list<const char*> problem) {
  for (const auto& kv : s.p)
    if (std::none_of(problem.begin(), problem.end(), [&](const char* key) { return kv.first == key; })) return false;
  return true;
}
static bool namesOnlyProduct(const KernelSpec& s) { return namesOnly(s, {"M", "N", "K", "BATCH", "TA", "TB", "ALIGN", "FILL", "OUT_BF16", "F16", "RELU", "SCALE_PTR"}); }

// GEMM whose wavefronts split k (kernels/gemm_wavek.hip).  type: 0 fp32, 1 bf16, 2 IEEE half, 3 fp8 e4m3.
struct WavekForm { int64_t tm, tn, vw, wk, depth; };

// Rows of whole 16-byte chunks (fp32: of four values and more; a 16-byte load of floats needs no more alignment than a float)
// whose offsets within a tile stay in 32 bits, and whole loads of a row-major B.
static bool wavekFits(const KernelSpec& s, int type, int64_t n, int64_t k) {
  const int64_t es = type == 0 ? 4 : type == 3 ? 1 : 2;
  return s.get("ALIGN", 0) >= 16 && shortRows(n, k) && k * es <= (1 << 24) && (type == 0 ? k >= 4 : k * es % 16 == 0) && !s.get("TA", 0) &&
         (type == 0 || s.get("TB", 0) || n * es % 16 == 0) && s.get("SCALE_PTR", 0) == 0;
}

bool emitGemmWavek(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err, int type, const WavekForm& f,
                   int64_t m, int64_t n, int64_t k, int64_t batch) {
  const int64_t es = type == 0 ? 4 : type == 3 ? 1 : 2;
  const bool tb = s.get("TB", 0) != 0;
  if (!wavekFits(s, type, n, k)) { err = s.family + ": WAVEK needs aligned operands (ALIGN = 16) in rows of whole 16-byte chunks, A contiguous along k"; return false; }
  if (f.tm < 1 || f.tm > 8 || f.tn < 1 || f.tn > 16 || f.wk < 1 || f.wk > 16 || f.depth < 1 || f.depth > 16 ||
      (!tb && (f.vw * es < 2 || f.vw * es > 16 || (f.vw & (f.vw - 1)) || f.tn % f.vw || n % f.vw))) {
    err = s.family + ": WAVEK is 1 to 16, TM 1 to 8, TN 1 to 16, DEPTH 1 to 16, and row-major weights need VW columns of 2 to 16 bytes that divide TN and N";
    return false;
  }
  // (every wavefront needs a k-step of its own)
  if (f.wk > ceilDiv(k * es, 128)) { err = s.family + ": WAVEK is at most the number of 128-byte steps along k"; return false; }
  if (f.wk * std::max((16 * f.tm + (tb ? 16 * f.tn : 0)) * 128, 16 * f.tm * (16 * f.tn + 4) * 4) > 160 * 1024) { err = s.family + ": the wavefronts' rows and partial sums need more than 160 KiB of LDS"; return false; }
  const bool out16 = s.get("OUT_BF16", 0) != 0;
  s.p["WAVEK"] = f.wk; s.p["TM"] = f.tm; s.p["TN"] = f.tn; s.p["DEPTH"] = f.depth;
  if (!tb) s.p["VW"] = f.vw;
  Defines d;
  d.add("GW_NAME", s.name);
  d.add("GW_M", m); d.add("GW_N", n); d.add("GW_K", k); d.add("GW_BATCH", batch);
  d.add("GW_TYPE", type);
  d.add("GW_OUT16", out16 ? 1 : 0);
  d.add("GW_TB", tb ? 1 : 0);
  d.add("GW_TM", f.tm); d.add("GW_TN", f.tn);
  if (!tb) d.add("GW_VW", f.vw);
  d.add("GW_WK", f.wk);
  d.add("GW_DEPTH", f.depth);
  d.add("GW_RELU", s.get("RELU", 0) ? 1 : 0);
  src = d.wrap(kTpl_gemm_wavek);
  info.name = s.name;
  info.grid[0] = (uint32_t)(ceilDiv(m, 16 * f.tm) * ceilDiv(n, 16 * f.tn));
  info.grid[1] = (uint32_t)batch;
  info.block[0] = (uint32_t)(64 * f.wk);
  info.numArgs = type == 3 ? 5 : 3;
  info.numScalars = type == 3 ? 2 : 0;
  info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
  info.bytes = (double)batch * ((double)es * ((double)m * k + (double)k * n) + (out16 ? 2.0 : 4.0) * (double)m * n);
  return true;
}

static WavekForm wavekAsked(const KernelSpec& s, int type) {
  return {s.get("TM", 1), s.get("TN", 4), s.get("VW", s.get("N", 0) % 4 || s.get("TN", 4) % 4 ? (type == 3 ? 2 : 1) : 4), s.get("WAVEK", 0), s.get("DEPTH", 2)};
}

// Time in us of a form whose wavefronts split k: a launch and the fixed parts of the kernel, then what is slowest of a compute
// unit's intake (MB), the card's (MB from memory, MB through the L2s) and the MFMAs, and on top the partial sums (tiles x
// wavefronts) and the steps that a wavefront waits for one after the other.  Fitted to 7000 timings of 200 products of the sizes
// that launches of few tiles have (linear layers of 1 to 700 rows, 512 to 11008 columns, K 512 to 4096; fp32 256 to 2048 a
// side, 1 to 16 of them): the form of least modelled time is within 3 % (k-contiguous B) to 7 % of the best on average.
struct WavekRates { double fixed, cu, hbm, sums, wait, l2, mfma, odd; };
static double wavekTime(int type, bool tb, bool out16, const WavekForm& f, int64_t m, int64_t n, int64_t k, int64_t batch) {
  static const WavekRates rates[3][2] = {      // row-major B, k-contiguous B; `odd`: fp32 rows that start off 16 bytes, intake
      {{2.35, 13.1, 0.41, 0.112, 0.024, 0.045, 1.55, 0.85}, {2.60, 8.25, 0.53, 0.131, 0.065, 0.018, 1.45, 1.24}},
      {{2.23, 12.5, 0.21, 0.227, 0.103, 0.052, 3.42, 0.0}, {1.95, 8.82, 0.153, 0.408, 0.106, 0.041, 3.15, 0.0}},
      {{2.40, 12.8, 0.267, 0.074, 0.127, 0.099, 2.97, 0.0}, {2.15, 10.2, 0.168, 0.220, 0.066, 0.047, 2.59, 0.0}}};
  const WavekRates& r = rates[type == 0 ? 0 : type == 3 ? 2 : 1][tb ? 1 : 0];
  const double es = type == 0 ? 4 : type == 3 ? 1 : 2, kb = (double)k * es;
  const double tiles = (double)ceilDiv(m, 16 * f.tm) * (double)ceilDiv(n, 16 * f.tn) * (double)batch, per = std::ceil(tiles / 256.0);
  const double rows = (double)std::min<int64_t>(16 * f.tm, ceilDiv(m, 8) * 8), bytes = (rows + 16.0 * f.tn) * kb;
  const double steps = std::ceil(std::ceil(kb / 128.0) / (double)f.wk);
  const double hbm = (kb * (double)(m + n) + (double)m * (double)n * (out16 ? 2.0 : 4.0)) * (double)batch;
  const double mfma = (type == 0 ? 256.0 : type == 3 ? 64.0 : 32.0) * f.tm * f.tn * steps * per * std::max(1.0, f.wk / 4.0) / 2400.0;
  // workgroups that a CU holds at a time: by LDS, and by registers (the slots, the sums, a set of fragments, addresses)
  const int64_t lds = f.wk * std::max((16 * f.tm + (tb ? 16 * f.tn : 0)) * 128, 16 * f.tm * (16 * f.tn + 4) * 4);
  const int64_t regs = ceilDiv(8 * f.depth * (f.tm + f.tn) + 4 * f.tm * f.tn + 8 * f.tm + 40, 8) * 8;
  const int64_t waves = std::max<int64_t>(1, std::min<int64_t>(8, 512 / regs)) * 4;
  const double held = (double)std::max<int64_t>(1, std::min<int64_t>(160 * 1024 / lds, waves / f.wk));
  const double wait = std::ceil(tiles / (256.0 * held)) * steps / std::min<double>((double)f.depth, std::max(1.0, steps));
  const double odd = type == 0 && k % 4 ? 1.0 + r.odd : 1.0;
  auto p4 = [](double x) { return x * x * x * x; };
  const double most = std::pow(p4(odd * r.cu * bytes * per / 1e6) + p4(odd * r.hbm * hbm / 1e6) + p4(odd * r.l2 * bytes * tiles / 1e6) + p4(r.mfma * mfma), 0.25);
  return r.fixed + most + r.sums * per * f.tm * f.tn * f.wk / 16.0 + r.wait * wait;
}

// Whether a form's registers hold it.  Eight wavefronts leave 256 each; beside 128 of slots and sums the compiler still finds room for
// fragments, addresses and the last steps that it unrolls, beside 160 not (up to 480 bytes a lane in scratch memory; 36 at 33 x 3840 x
// 2816 fp8 row-major on 64 x 32 tiles, two steps in flight), nor beside 64 sums while it sorts a row-major B of 8 or 16 bits.  The next
// best forms are 1.29 (fp8, 13 products whose form spilled) and 1.16 (fp32, 17) times as fast: 63 x 7072 x 3712 fp8 20.1 us and
// 10.6, 320 x 901 x 3205 fp32 66.7 and 51.2; those that did not spill gain 3 % on average
// and lose 9 % at worst (fp8 33 x 3856 x 2880 7.1 and 7.7).
static bool wavekStaysInRegisters(int type, bool tb, const WavekForm& f) {
  const int64_t es = type == 0 ? 4 : type == 3 ? 1 : 2;
  const int64_t slotB = tb ? 8 * f.tn : 2 * f.tn / f.vw * (16 / es) * std::max<int64_t>(1, f.vw * es / 4);
  return f.wk <= 4 || (f.depth * (8 * f.tm + slotB) + 4 * f.tm * f.tn <= 128 && (tb || type == 0 || f.tm * f.tn < 16));
}

// The form of least modelled time, if there is one and the caller asks for it (FILL = 2); `us`: that time.
static bool chooseWavek(const KernelSpec& s, int type, int64_t m, int64_t n, int64_t k, int64_t batch, WavekForm& best, double& us) {
  if (s.get("FILL", 0) < 2 || !wavekFits(s, type, n, k)) return false;
  static const int64_t tiles[][2] = {{1, 1}, {1, 2}, {2, 1}, {2, 2}, {1, 4}, {2, 4}, {4, 2}, {4, 4}, {3, 4}, {4, 3}};
  const bool tb = s.get("TB", 0) != 0, out16 = s.get("OUT_BF16", 0) != 0;
  const int64_t es = type == 0 ? 4 : type == 3 ? 1 : 2, steps = ceilDiv(k * es, 128);
  us = 0.0;
  for (const auto& t : tiles) {
    const bool thirds = t[0] == 3 || t[1] == 3;
    if ((thirds && type != 0) || (t[0] > 1 && 8 * t[0] >= m)) continue;
    if (!tb && type == 3 && t[1] < 2) continue;                                    // loads of two columns and more
    if (t[0] == 1 && t[1] == 4 && (tb || type != 3)) continue;
    if (t[1] == 1 && t[0] == 2 && !tb) continue;
    for (int64_t wk : {4, 8})
      for (int64_t depth : {1, 2}) {
        if (wk > steps || (depth > 1 && steps <= wk)) continue;
        const WavekForm f = {t[0], t[1], tb ? 1 : n % 4 || t[1] % 2 ? 1 : std::min<int64_t>(t[1], 4), wk, depth};
        if (!wavekStaysInRegisters(type, tb, f)) continue;
        const double time = wavekTime(type, tb, out16, f, m, n, k, batch);
        if (us == 0.0 || time < us) { us = time; best = f; }
      }
  }
  return us > 0.0;
}

bool emitGemmF32(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  int64_t m, n, k, batch;
  if (!gemmCommon(s, err, m, n, k, batch)) return false;
  if (s.get("WAVEK", 0) > 0) return emitGemmWavek(s, src, info, err, 0, wavekAsked(s, 0), m, n, k, batch);
  // The largest square tile that still gives every CU a workgroup (measured on 4096^3, 2048^3, 1024^3 and
  // 16 x 1024^3: 256^2 with 16 wavefronts, 128^2 with 16 and a deeper k-tile, 64^2 with 4 and a deeper k-tile).
  int64_t tile = 64;
  for (int64_t t : {256, 128}) {
    if (m < t || n < t) continue;
    if ((double)ceilDiv(m, t) * (double)ceilDiv(n, t) * (double)batch >= 256.0) { tile = t; break; }
  }
  // Sizes that this tile does not divide, and a B contiguous along k for the direct loads, get the tile of least work instead:
  // rounds of 256 tiles times the tile's area, weighted by the rate it reaches (4000 x 4096 x 4096: 256 912 us, 128 928, 64
  // 971).  The last tiles are moved back (no guards), so small tiles cost little and leave little idle.  Direct loads need rows
  // of whole 16-byte chunks and a caller who has looked at the operands' addresses (ALIGN = 16); us, against guarded 256 or 128
  // tiles: 16 x 777 x 1000 x 500 118 and 167, 2 x 1100 x 1300 x 900 50 and 65, 1500 x 2048 x 300 19 and 24; 2048 x 1984 x
  // 1088 takes 128: 68 and 78.  Rows of any length, through registers: 1501 x 2047 x 303 21 and 31, 777 x 1003 x 501 13 and 23.
  // k-tiles of 32 for 64 x 64 direct-load tiles whose rows are then whole 128-byte lines (1024^3 with a k-contiguous B: 18.8
  // us, 16 21.4), else of 16 (K 500, 777 x 1000: 16 11.8 us, 32 20.4: every row of a k-tile of 32 straddles two lines).
  bool own = false;
  for (const char* key : {"BM", "BN", "BK", "WM", "WN", "WK", "NBUF", "PAD"}) own = own || s.has(key);
  const bool direct = s.get("D2L", 1) != 0 && s.get("ALIGN", 0) >= 16 && shortRows(n, k) && !s.get("TA", 0) && k % 4 == 0 && (s.get("TB", 0) || n % 4 == 0);
  const bool plain = namesOnlyProduct(s);
  const bool divides = m % tile == 0 && n % tile == 0 && k % (tile <= 128 ? 32 : 16) == 0;
  if (!own && (!divides || (direct && s.get("TB", 0))) && m >= 64 && n >= 64 && k >= 16) {
    static const struct { int64_t t; double weight; } sizes[] = {{256, 0.985}, {128, 1.0}, {64, 1.06}};
    double least = 0.0;
    for (const auto& z : sizes) {
      if (m < z.t || n < z.t) continue;
      const double work = std::ceil((double)ceilDiv(m, z.t) * (double)ceilDiv(n, z.t) * (double)batch / 256.0) * (double)(z.t * z.t) * z.weight;
      if (least == 0.0 || work < least) { least = work; tile = z.t; }
    }
    s.p["BM"] = s.p["BN"] = tile;
    s.p["BK"] = direct ? (tile == 64 && k % 32 == 0 ? 32 : 16) : (tile == 128 ? 32 : 16);
    s.p["WM"] = s.p["WN"] = tile == 64 ? 2 : 4;
    if (s.get("TB", 0)) { s.p["WK"] = 1; s.p["NBUF"] = 2; }    // two wavefront groups gain nothing where B is read 16 bytes at a time (19.9 us at 1024^3)
  }
  // Few tiles: wavefronts that split k, where the models say so clearly.  This kernel's time (fitted to the same products, within 12 %
  // on average): rounds of tiles and the part of them in use, and on few 64 x 64 tiles a k-tile's way from memory.  us, this and
  // that: 256^3 6.6 and 2.5, 256 x 256 x 2048 36 and 7.1, 2 x 700 x 300 x 1500 47 and 20; 1500 x 400 x 1100 34 and 22; level at
  // 1024^3 (20); 4 x 1024^3 70 and 75.
  if (plain && m >= 64 && n >= 64 && k >= 16) {
    WavekForm form;
    double us;
    if (chooseWavek(s, 0, m, n, k, batch, form, us)) {
      const double groups = (double)ceilDiv(m, tile) * (double)ceilDiv(n, tile) * (double)batch, rounds = std::ceil(groups / 256.0);
      const double area = (double)(tile * tile) / 4096.0, used = std::max(0.3, groups / 256.0), sparse = tile == 64 ? std::max(0.0, 1.0 - groups / 512.0) : 0.0;
      const double tiled = s.get("TB", 0) ? 2.95 + 0.01 * k * (area * (1.044 * rounds + 0.681 * used) * (direct ? 1.0 : 1.33) + 0.68 * sparse)
                                          : 3.07 + 0.01 * k * (area * (1.454 * rounds + 0.239 * used) * (direct ? 1.0 : 1.26) + 0.32 * sparse);
      // (k-contiguous B on whole k-tiles of 32 is faster than modelled: 3 x 532 x 388 x 1184 22.2 us, split 23.6)
      if (us < (s.get("TB", 0) && direct && k % 32 == 0 ? 0.8 : 0.88) * tiled) return emitGemmWavek(s, src, info, err, 0, form, m, n, k, batch);
    }
  }
  int64_t bm = s.get("BM", tile), bn = s.get("BN", tile);
  int64_t bk = s.get("BK", bm <= 128 && bn <= 128 ? 32 : 16);
  int64_t wm = s.get("WM", bm >= 128 ? 4 : 2), wn = s.get("WN", bn >= 128 ? 4 : 2), gm = s.get("GROUP_M", 8);
  if (!checkTile(s, bm, bn, bk, wm, wn, 4, err)) return false;
  const int64_t pad = s.get("PAD", 4);
  if (pad < 0 || pad % 4) { err = "gemm_f32: PAD must be a multiple of 4 floats"; return false; }
  const int64_t lds = 2 * bk * ((bm + pad) + (bn + pad)) * 4;
  if (lds > 160 * 1024) { err = "gemm_f32: tile needs more than 160 KiB of LDS"; return false; }
  const bool edge = (m % bm) || (n % bn) || (k % bk);
  s.p["BM"] = bm; s.p["BN"] = bn; s.p["BK"] = bk; s.p["WM"] = wm; s.p["WN"] = wn; s.p["GROUP_M"] = gm;

  // Whole tiles with BK = 16 or 32 of two row-major operands: the kernel that loads both tiles straight into LDS
  // (kernels/gemm_f32_d2l.hip).  Where the caller has looked at the operands' addresses (ALIGN = 16) and rows are whole
  // 16-byte chunks, also a B that is contiguous along k, and sizes that the tiles do not divide.
  const bool aligned = s.get("ALIGN", 0) >= 16 && shortRows(n, k) && k % 4 == 0 && (s.get("TB", 0) || n % 4 == 0) && m >= bm && n >= bn && k >= bk;
  const bool d2l = s.get("D2L", 1) != 0 && !s.get("TA", 0) && (!s.get("TB", 0) || aligned) && (bk == 16 || bk == 32) && (!edge || aligned) && bm % 64 == 0 &&
                   (bn == 64 || bn == 128 || bn == 256) && bm % (32 * wm) == 0 && bn % (32 * wn) == 0 && (bm + bn) * bk * 8 <= 160 * 1024;
  s.p["D2L"] = d2l;
  // WK = 2: two groups of WM x WN wavefronts split the steps of every k-tile and add their partial sums through LDS at
  // the end (the kernel says why); needs k-tiles of 32, at most 16 wavefronts in all and results that fit the LDS tiles
  const bool wkFits = d2l && bk == 32 && wm * wn * 2 <= 16 && bm * bn * 4 <= (bm + bn) * bk * 8;
  // 64 x 64 x 32 tiles of four wavefronts on a launch that gives a CU at most one workgroup: two groups and three buffers
  // (1024^3: 19.7 against 20.7-21.1 us, 512 x 512 x 2048: 35.6 against 37.8 us; either one alone is slower, 22.5 and 23.7 us;
  // with several workgroups per CU, 1536^3, the groups change nothing and the launch keeps the plain form)
  const bool small = wkFits && bm == 64 && bn == 64 && wm * wn == 4 && ceilDiv(m, bm) * ceilDiv(n, bn) * batch <= 256;
  const int64_t wk = s.get("WK", small ? 2 : 1);
  if (wk != 1 && !(wk == 2 && wkFits)) { err = "gemm_f32: WK is 1 or 2; 2 needs the direct loads into LDS (D2L), BK = 32, at most eight wavefronts per group and BM * BN <= 64 (BM + BN)"; return false; }
  s.p["WK"] = wk;
  // NBUF LDS buffers per operand (the loads of k-tile kt + NBUF - 1 start with k-tile kt): more than two where a k-tile is
  // shorter than a load's way from the L2; every wavefront must then issue the same number of loads per k-tile
  const int64_t nbuf = s.get("NBUF", small && wk == 2 ? 3 : 2);
  const int64_t blocks = (bm + bn) * bk * 4 / 1024;
  if (nbuf != 2 && !(d2l && (nbuf == 3 || nbuf == 4) && blocks % (wm * wn * wk) == 0 && nbuf * (bm + bn) * bk * 4 <= 160 * 1024)) {
    err = "gemm_f32: NBUF is 2, or 3 or 4 with the direct loads into LDS (D2L) where a k-tile is a whole number of 1 KiB blocks per wavefront and fits the LDS that many times";
    return false;
  }
  s.p["NBUF"] = nbuf;
  if (d2l) {
    Defines d;
    d.add("GL_NAME", s.name);
    d.add("GL_M", m); d.add("GL_N", n); d.add("GL_K", k); d.add("GL_BATCH", batch);
    d.add("GL_BM", bm); d.add("GL_BN", bn); d.add("GL_BK", bk); d.add("GL_WM", wm); d.add("GL_WN", wn);
    d.add("GL_WK", wk);
    d.add("GL_NBUF", nbuf);
    d.add("GL_GROUP_M", gm);
    d.add("GL_RELU", s.get("RELU", 0) ? 1 : 0);
    if (m % bm || n % bn) d.add("GL_SHIFT", 1);
    if (k % bk) d.add("GL_KTAIL", 1);
    if (s.get("TB", 0)) d.add("GL_TB", 1);
    src = d.wrap(kTpl_gemm_f32_d2l);
    info.name = s.name;
    info.grid[0] = (uint32_t)(ceilDiv(m, bm) * ceilDiv(n, bn));
    info.grid[1] = (uint32_t)batch;
    info.block[0] = (uint32_t)(64 * wm * wn * wk);
    info.numArgs = 3;
    info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
    info.bytes = 4.0 * (double)batch * ((double)m * k + (double)k * n + (double)m * n);
    return true;
  }

  Defines d;
  d.add("GM_NAME", s.name);
  d.add("GM_M", m); d.add("GM_N", n); d.add("GM_K", k); d.add("GM_BATCH", batch);
  d.add("GM_TA", s.get("TA", 0) ? 1 : 0); d.add("GM_TB", s.get("TB", 0) ? 1 : 0);
  d.add("GM_BM", bm); d.add("GM_BN", bn); d.add("GM_BK", bk);
  d.add("GM_WM", wm); d.add("GM_WN", wn); d.add("GM_GROUP_M", gm);
  // Ragged sizes that hold a whole tile: the last tiles are moved back (any row length: a 16-byte load of floats needs an
  // alignment of four bytes, which every float has)
  const bool shift = edge && m >= bm && n >= bn;
  d.add("GM_EDGE", edge && !shift ? 1 : 0);
  if (shift) d.add("GM_SHIFT", 1);
  s.p["SHIFT"] = shift;
  d.add("GM_RELU", s.get("RELU", 0) ? 1 : 0);
  d.add("GM_PAD", pad);
  src = d.wrap(kTpl_gemm_f32);

  info.name = s.name;
  info.grid[0] = (uint32_t)(ceilDiv(m, bm) * ceilDiv(n, bn));
  info.grid[1] = (uint32_t)batch;
  info.block[0] = (uint32_t)(64 * wm * wn);
  info.numArgs = 3;
  info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
  info.bytes = 4.0 * (double)batch * ((double)m * k + (double)k * n + (double)m * n);
  return true;
}

// Default workgroup tile of the bf16 and fp8 GEMMs: the largest of 256x256, 128x128, 128x64 and 64x64 that still
// gives each of the 256 CUs a workgroup (measured on 1024^3 ... 8192^3, 512x4096x4096 and 4096x4096x512: the
// choice is within a few per cent of the best tile everywhere, where a fixed 256x256 loses up to 2x on 2048^3).
static void defaultGemmTile(int64_t m, int64_t n, int64_t batch, int64_t& bm, int64_t& bn) {
  static const int64_t cand[4][2] = {{256, 256}, {128, 128}, {128, 64}, {64, 64}};
  bm = bn = 64;
  for (const auto& c : cand)
    if ((double)ceilDiv(m, c[0]) * (double)ceilDiv(n, c[1]) * (double)batch >= 256.0) {
      bm = c[0];
      bn = c[1];
      return;
    }
}

// fp64 GEMM on v_mfma_f64_16x16x4_f64.  128 x 128 x 16 tiles; 64 x 64 tiles where the larger ones would leave
// compute units without a workgroup.
bool emitGemmF64(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  int64_t m, n, k, batch;
  if (!gemmCommon(s, err, m, n, k, batch)) return false;
  // measured at 4096^3 with 16 wavefronts: 128 x 256 tiles 68 TF (0.87 of the 78.6 TF peak), 256 x 128 66 TF,
  // 128 x 128 63.5 TF, 64 x 64 (four wavefronts) 54 TF; k-tiles of 8 or 32 instead of 16: 55 TF
  static const int64_t cand[3][2] = {{128, 256}, {128, 128}, {64, 64}};
  int64_t tm = 64, tn = 64;
  for (const auto& c : cand)
    if (m >= c[0] && n >= c[1] && (double)ceilDiv(m, c[0]) * (double)ceilDiv(n, c[1]) * (double)batch >= 256.0) { tm = c[0]; tn = c[1]; break; }
  int64_t bm = s.get("BM", tm), bn = s.get("BN", s.has("BM") ? s.get("BM", tn) : tn), bk = s.get("BK", 16);
  // wavefronts of 32 x 32 results (four MFMA tiles): 16 of them on a 128 x 128 tile measured 63 TF at 4096^3, 0.81
  // of the 78.6 TF peak, where four wavefronts of 64 x 64 reach 44 TF (one wavefront per SIMD hides no latency)
  int64_t wm = s.get("WM", std::max<int64_t>(1, std::min<int64_t>(4, bm / 32)));
  int64_t wn = s.get("WN", std::max<int64_t>(1, std::min<int64_t>(4, bn / 32))), gm = s.get("GROUP_M", 8);
  if (wm < 1 || wn < 1 || wm * wn > 16 || bm <= 0 || bn <= 0 || bm % (16 * wm) || bn % (16 * wn) || bk < 8 || bk % 8) {
    err = "gemm_f64: tile BM/BN must be multiples of 16*WM / 16*WN and BK a multiple of 8";
    return false;
  }
  if ((bm / wm / 16) * (bn / wn / 16) > 24) { err = "gemm_f64: more than 24 MFMA tiles per wavefront do not fit the registers"; return false; }
  const int64_t lds = 2 * (bm + bn) * (bk + 2) * 8;      // both tiles with k innermost, rows of BK + 2 doubles
  if (lds > 160 * 1024) { err = "gemm_f64: tile needs more than 160 KiB of LDS"; return false; }
  const bool edge = (m % bm) || (n % bn) || (k % bk);
  s.p["BM"] = bm; s.p["BN"] = bn; s.p["BK"] = bk; s.p["WM"] = wm; s.p["WN"] = wn; s.p["GROUP_M"] = gm;

  // Whole tiles with BK = 16 of two row-major operands: the kernel that loads both tiles straight into LDS
  // (kernels/gemm_f64_d2l.hip)
  const bool d2l = s.get("D2L", 1) != 0 && !s.get("TA", 0) && !s.get("TB", 0) && bk == 16 && !edge && bm % 64 == 0 && (bn == 128 || bn == 256) &&
                   bm % (16 * wm) == 0 && bn % (32 * wn) == 0 && 2 * (bm * 128 + 16 * bn * 8) <= 160 * 1024;
  s.p["D2L"] = d2l;
  if (d2l) {
    Defines d;
    d.add("GE_NAME", s.name);
    d.add("GE_M", m); d.add("GE_N", n); d.add("GE_K", k); d.add("GE_BATCH", batch);
    d.add("GE_BM", bm); d.add("GE_BN", bn); d.add("GE_WM", wm); d.add("GE_WN", wn);
    d.add("GE_GROUP_M", gm);
    d.add("GE_RELU", s.get("RELU", 0) ? 1 : 0);
    src = d.wrap(kTpl_gemm_f64_d2l);
    info.name = s.name;
    info.grid[0] = (uint32_t)((m / bm) * (n / bn));
    info.grid[1] = (uint32_t)batch;
    info.block[0] = (uint32_t)(64 * wm * wn);
    info.numArgs = 3;
    info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
    info.bytes = 8.0 * (double)batch * ((double)m * k + (double)k * n + (double)m * n);
    return true;
  }

  Defines d;
  d.add("GD_NAME", s.name);
  d.add("GD_M", m); d.add("GD_N", n); d.add("GD_K", k); d.add("GD_BATCH", batch);
  d.add("GD_TA", s.get("TA", 0) ? 1 : 0); d.add("GD_TB", s.get("TB", 0) ? 1 : 0);
  d.add("GD_BM", bm); d.add("GD_BN", bn); d.add("GD_BK", bk);
  d.add("GD_WM", wm); d.add("GD_WN", wn); d.add("GD_GROUP_M", gm);
  d.add("GD_EDGE", edge ? 1 : 0);
  d.add("GD_RELU", s.get("RELU", 0) ? 1 : 0);
  src = d.wrap(kTpl_gemm_f64);

  info.name = s.name;
  info.grid[0] = (uint32_t)(ceilDiv(m, bm) * ceilDiv(n, bn));
  info.grid[1] = (uint32_t)batch;
  info.block[0] = (uint32_t)(64 * wm * wn);
  info.numArgs = 3;
  info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
  info.bytes = 8.0 * (double)batch * ((double)m * k + (double)k * n + (double)m * n);
  return true;
}

// Tail split of a tiled GEMM (see kernels/gemm_bf16.hip): SK_UNITS extra workgroups share the k-iterations of
// the tiles behind the first SK_FULL ones and leave partial sums in a workspace.  Only on request (SK_UNITS > 0):
// on the 4096 x 11008 x 4096 product it measured slower than one workgroup per tile (0.53 against 0.34 ms).  The
// tiles of a round that run side by side read the same A and B panels at the same k and share them in the L2;
// runs that start at different k read their operands alone.  And the partly filled last round costs little to
// begin with: 256, 512 and 688 workgroups of that kernel take 0.123, 0.242 and 0.343 ms, the last 176 tiles
// 0.100 ms on CUs that then have more of the chip's power and bandwidth each.
bool chooseTailSplit(const KernelSpec& s, int64_t tiles, int64_t kt, int64_t batch, int64_t& full, int64_t& units,
                     std::string& err) {
  full = 0;
  units = s.get("SK_UNITS", 0);
  if (units <= 0) {
    units = 0;
    return true;
  }
  full = s.get("SK_FULL", tiles / units * units == tiles ? tiles - units : tiles / units * units);
  const int64_t tail = tiles - full;
  const bool xcd = units % 8 == 0 && full % 8 == 0 && tail % 8 == 0 && tiles % 8 == 0;
  const int64_t groups = xcd ? 8 : 1;
  int64_t per = ceilDiv((tail / groups) * kt, units / groups);
  per += per & 1;      // whole pairs of k-iterations: the kernel's k loop runs in pairs
  if (batch != 1 || units > 4096 || full < 0 || tail < 1 || tail > 1024 || per > kt || kt % 2) {
    err = s.family + ": tail split needs one batch, 1..1024 tail tiles, an even number of k-tiles and at most one tile's "
                     "k-iterations per unit";
    return false;
  }
  return true;
}

// Tile, wavefronts and LDS buffers of a 16-bit GEMM with direct loads: the least modelled time of the forms below.  A
// form's workgroups run `slots` at a time (one or two per CU, by their LDS); a round of them takes a + b * (share of the
// slots in use), in us at K = 4096, fitted to 400 timings of both weight layouts (M 1-4001, N 1024-11008, K 1024-4096;
// the choice is within 10 % of the best form on all but two of 28 shapes, and there within 15 %).  Examples, us:
//   M, N, K            256x256/2  128x128/2  128x128/3  64x128/3  64x128/4  64x64/4      (tile / LDS buffers)
//   4001, 11008, 4096     284        351                                      795
//   1000, 11008, 4096      87         97         92       107       119       124
//    300, 11008, 4096      75         45         55        38        40        45
//    512,  4096, 4096      75         40         25        23        22        25
//    128,  4096, 4096                 40         24        21        18        13
//     16, 11008, 4096                                      21        18        15
// A small tile has few MFMAs per k-tile to hide a load under: with two buffers (one k-tile ahead) the 128 x 4096 x 4096
// product waits 0.45 us per k-tile, with four 0.2.
struct Gemm16Form { int64_t bm, bn, wm, wn, nbuf; double slots, a, b; };
static const Gemm16Form* chooseGemm16Form(int64_t m, int64_t n, int64_t k, int64_t batch, double* modelled = nullptr) {
  static const Gemm16Form forms[] = {
      {256, 256, 4, 2, 2, 256, 55, 45}, {128, 128, 4, 2, 2, 512, 32, 31}, {128, 128, 4, 2, 3, 256, 14, 25},
      {64, 128, 2, 2, 3, 512, 13, 28},  {64, 128, 2, 2, 4, 256, 18, 5},   {64, 64, 2, 2, 4, 512, 12, 12},
  };
  // few rows: tiles of 32 x 64 (us, against 64 x 64: 8 x 1024 x 4096 9.2 and 11.6, 16 x 11008 x 4096 14.6 and 15.0, 32 x 4096 x
  // 4096 12.1 and 13.2, 1 x 4096 x 4096 11.4 and 12.3)
  static const Gemm16Form few = {32, 64, 1, 4, 4, 512, 0, 0};
  if (modelled) *modelled = 0.0;
  if (m <= 32 && batch == 1 && n >= 64 && k >= 64) return &few;
  const Gemm16Form* best = nullptr;
  double least = 0.0;
  for (const auto& f : forms) {
    if ((m < f.bm && (f.bm > 64 || batch != 1)) || n < f.bn || k < 64) continue;
    // a moved-back k-tile costs this form up to 128 bytes of scratch a lane: 1500 x 11008 x 1040 70 us against 61 in 128 x 128 tiles,
    // x 1104 68 against 65, x 4080 198 against 195; many rounds would gain all the same, 4001 x 11008 x 4072 492 against 325
    if (k % 64 && f.bm == 256) continue;
    const double tiles = (double)ceilDiv(m, f.bm) * (double)ceilDiv(n, f.bn) * (double)batch, rounds = std::ceil(tiles / f.slots);
    if (f.bn == 128 && f.nbuf == 4 && rounds > 1) continue;     // one workgroup per CU pays in a single round only
    const double cost = rounds * (f.a + f.b * tiles / (rounds * f.slots));
    if (!best || cost < least) { best = &f; least = cost; }
  }
  if (modelled) *modelled = least;
  return best;
}

// Tiles with a side of 192: where 256 or 128 a side leave the last round of workgroups nearly empty, the sizes between them fill it.
// The form of least modelled time among them if it is ahead of all the tiles above, else `form`.  Modelled as above, all forms
// fitted anew to 1000 timings of 93 products of 128 to 4096 rows (10 to 16 % off each): of those the choice takes 28, 12 % faster on
// average and 4 % slower at worst.  us, without and with: 1000 x 11008 x 4096 103 and 89, row-major 90 and 83; 400 x 11008 x 4096 69
// and 51; 1500 x 11008 x 4096 172 and 148; 3000 x 5504 x 1536 72 and 55; 4096 x 11008 x 4096 stays, 298 against 338.
static const Gemm16Form* chooseThirds(const Gemm16Form* form, int64_t m, int64_t n, int64_t k, int64_t batch) {
  static const Gemm16Form forms[] = {
      {256, 192, 4, 2, 2, 256, 68.6, 17.0}, {192, 256, 2, 4, 2, 256, 68.7, 18.5}, {128, 192, 4, 2, 2, 512, 46.9, 45.7},
      {128, 192, 4, 2, 3, 256, 37.1, 12.4}, {192, 128, 2, 4, 2, 512, 49.4, 43.9}, {192, 128, 2, 4, 3, 256, 40.3, 9.3},
      {256, 256, 4, 2, 2, 256, 81.5, 20.8}, {128, 128, 4, 2, 2, 512, 39.2, 27.0}, {128, 128, 4, 2, 3, 256, 26.8, 9.5},
      {64, 128, 2, 2, 3, 512, 17.8, 25.8},  {64, 128, 2, 2, 4, 256, 21.6, 3.6}};
  // (a moved-back k-tile among few: 3116 x 6032 x 528 39 and 45)
  if (!form || form->bm < 64 || m < 128 || (k % 64 && k < 1024)) return form;
  const Gemm16Form* best = nullptr;
  double least = 0.0;
  for (const auto& f : forms) {
    if (m < f.bm || n < f.bn || (k % 64 && f.bm == 256)) continue;
    const double tiles = (double)ceilDiv(m, f.bm) * (double)ceilDiv(n, f.bn) * (double)batch;
    const double us = 2.5 + (double)k / 4096.0 * (std::ceil(tiles / f.slots) * f.a + tiles / f.slots * f.b);
    if (!best || us < least) { best = &f; least = us; }
  }
  return best && (best->bm == 192 || best->bn == 192) ? best : form;
}

// Whether wavefronts that split k take less time than `tiled`, the form chosen above with `cost`: its time, fitted to the same
// products as wavekTime (within 8 to 14 %), from that cost, or for 32-row tiles from their number.  us, this and that: bf16
// k-contiguous 8 x 1024 x 4096 8.9 and 4.1, 16 x 2048 x 2048 5.6 and 3.3, 16 x 4096 x 4096 11.5 and 7.2, 64 x 1024 x 4096 12.8 and
// 5.4, 200 x 1024 x 4096 13.3 and 8.7; but 64 x 11008 x 4096 22.1 against 21.3, 200 x 4096 x 1024 6.2 against 7.1.  fp8 row-major
// 16 x 4096 x 4096 17.9 and 8.8.
static bool wavekAhead(const KernelSpec& s, int type, const Gemm16Form* tiled, double cost, int64_t m, int64_t n, int64_t k, int64_t batch, WavekForm& form) {
  double us;
  if (!tiled || !chooseWavek(s, type, m, n, k, batch, form, us)) return false;
  static const struct { double few0, few1, few2, hbm, many0, many1; } fits[2][2] = {     // 16 bits, fp8; row-major B, k-contiguous
      {{1.95, 8.75, 0.0326, 0.0, 2.61, 1.124}, {2.13, 6.60, 0.0447, 0.0, 3.0, 0.897}},
      {{1.55, 19.0, 0.141, 0.0, 2.88, 1.914}, {2.17, 9.54, 0.0145, 0.197, 2.44, 1.31}}};
  const auto& c = fits[type == 3][s.get("TB", 0) ? 1 : 0];
  const double es = type == 3 ? 1 : 2, depth = (double)k * es / 8192.0, hbm = c.hbm * (double)(m + n) * (double)k * es / 1e6;
  const double chain = depth * (c.few1 + c.few2 * (double)ceilDiv(n, 64));
  const double time = tiled->bm == 32 ? c.few0 + std::pow(chain * chain * chain * chain + hbm * hbm * hbm * hbm, 0.25) : c.many0 + c.many1 * depth * cost;
  // What is asked of the models: 10 % for small tiles; 20 % for large ones, which near a full round of 256 are up to 18 % slower
  // than modelled (1000 x 1024 x 4096 bf16 16.9, tiles 14.5); 30 % against whole fp8 tiles, which are faster than modelled.
  // Over 560 products of 1 to 1500 rows the choice is then 1.22 times as fast as tiles alone, and 7 % slower at worst.
  const bool wholeFp8 = type == 3 && m % 64 == 0 && n % 64 == 0 && k % 128 == 0;
  return us < (wholeFp8 ? 0.7 : form.tm * form.tn >= 8 ? 0.8 : 0.9) * time;
}

bool emitGemmBf16(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  int64_t m, n, k, batch;
  if (!gemmCommon(s, err, m, n, k, batch)) return false;
  if (s.get("WAVEK", 0) > 0) return emitGemmWavek(s, src, info, err, s.get("F16", 0) ? 2 : 1, wavekAsked(s, s.get("F16", 0) ? 2 : 1), m, n, k, batch);
  // Where the caller has looked at the operands' addresses (ALIGN = 16) and asks for no tile or switch of its own, and every
  // row starts on 16 bytes: one of the forms with direct loads
  bool own = false;
  for (const char* key : {"BM", "BN", "BK", "WM", "WN", "M16", "D2L", "BTR", "BPAD", "STAGES", "NBUF", "SK_UNITS", "INTERLEAVE", "SETPRIO"}) own = own || s.has(key);
  const Gemm16Form* form = nullptr;
  if (!own && s.get("ALIGN", 0) >= 16 && shortRows(n, k) && !s.get("TA", 0) && k % 8 == 0 && (s.get("TB", 0) || n % 8 == 0)) {
    double cost;
    form = chooseGemm16Form(m, n, k, batch, &cost);
    WavekForm split;
    const int type = s.get("F16", 0) ? 2 : 1;
    if (namesOnlyProduct(s) && wavekAhead(s, type, form, cost, m, n, k, batch, split)) return emitGemmWavek(s, src, info, err, type, split, m, n, k, batch);
    if (!s.get("FP8_PAIRS", 0)) form = chooseThirds(form, m, n, k, batch);
  }
  if (form) {
    s.p["BM"] = form->bm; s.p["BN"] = form->bn; s.p["WM"] = form->wm; s.p["WN"] = form->wn;
    s.p["M16"] = 1; s.p["D2L"] = 1; s.p["NBUF"] = form->nbuf;
  }
  int64_t dm, dn;
  defaultGemmTile(m, n, batch, dm, dn);
  int64_t bm = s.get("BM", dm);
  int64_t bn = s.get("BN", dn);
  int64_t bk = s.get("BK", 64);
  // 256x256 tiles run as 8 wavefronts (two per SIMD, 64x128 each) so that one wavefront's
  // LDS and global-memory instructions issue under the other's MFMAs
  int64_t wm = s.get("WM", bm >= 256 && bn >= 256 ? 4 : 2), wn = s.get("WN", 2), gm = s.get("GROUP_M", 8);
  // an A tile of 32 rows, four wavefronts side by side: direct loads of at most so many rows only (checked below)
  const bool fewRows = bm == 32 && bn == 64 && wm == 1 && wn == 4 && bk == 64 && m <= bm && batch == 1 && s.get("M16", 0) && s.get("D2L", 1);
  if (!fewRows && !checkTile(s, bm, bn, bk, wm, wn, 16, err)) return false;
  // A tiles k-contiguous with 16 bytes of padding a row; B tiles the same, or [k][n] rows with 32 bytes of padding
  // pad of an sB[k][n] row: the 32 lanes that a transposing read serves together take four k rows of 64 bytes, which fall
  // on disjoint banks when the row pitch is 64 modulo 256 (SQ_LDS_BANK_CONFLICT: 22.5 M cycles per launch of the
  // 4096 x 11008 x 4096 product with a pad of 32, none with 64)
  int64_t bpad = s.get("BPAD", (bn * 2) % 256 == 0 ? 64 : 32);
  if (bpad < 0 || bpad % 16) { err = "gemm_bf16: BPAD must be a multiple of 16 bytes"; return false; }
  const bool ragged = (m % bm) || (n % bn) || (k % bk) || fewRows;
  // Ragged sizes without guarded loads: the last tiles are moved back to end at the edge (GB_SHIFT in the kernel).  Needs a
  // whole tile in every dimension, rows that start on 16-byte boundaries (ALIGN = 16: the caller has looked at the
  // operands' addresses; without it the guarded loads, which take any address, stay) and no tail split.
  // fewer rows than one tile: the rows past the last are read from the last one (GB_CLAMP; direct loads only)
  // (tiles of at most 64 rows: a lane's 32-bit offset spans the rows of the tile, and the whole-row epilogue of the 256 x 256
  // tile stores every row that it holds)
  const bool clamp = ((m < bm && bm <= 64) || fewRows) && batch == 1 && s.get("D2L", 1) != 0;
  const bool canShift = s.get("ALIGN", 0) >= 16 && shortRows(n, k) && (m >= bm || clamp) && n >= bn && k >= bk && k % 8 == 0 && (!s.get("TA", 0) || m % 8 == 0) &&
                        (s.get("TB", 0) || n % 8 == 0) && s.get("SK_UNITS", 0) <= 0;
  // the 16x16x32 MFMA (see the kernel): whole 64-deep k-tiles, A contiguous along k, B contiguous along k or read
  // through the transposing LDS reads, loads without guards
  const bool m16Fits = bk == 64 && !s.get("TA", 0) && (s.get("TB", 0) || s.get("BTR", 1)) && (!ragged || canShift) &&
                       (wm * wn) % 2 == 0 && (fewRows || bm % (8 * wm * wn) == 0) && bn % (8 * wm * wn) == 0 && s.get("STAGES", 1) == 1 &&
                       s.get("SK_UNITS", 0) <= 0 && bm / wm % 16 == 0 && bn / wn % 16 == 0;
  // direct loads into LDS (global_load_lds_dwordx4, see the kernel): every wavefront moves a whole, even number of
  // 1 KiB blocks per operand tile; row-major weights need the 256-column tile and eight wavefronts
  const int64_t waves = wm * wn;
  auto evenBlocks = [&](int64_t side) { return side % (16 * waves) == 0 || (side == 192 && waves == 8); };   // (192: three blocks each)
  const bool d2lFits = m16Fits && (fewRows ? canShift : evenBlocks(bm)) &&
                       (s.get("TB", 0) ? evenBlocks(bn) : ((bn == 64 || bn == 128 || bn == 192 || bn == 256) && (bn / 8) % waves == 0));
  // Default on the 256 x 256 tile with eight wavefronts, where it was measured: with direct loads 0.295-0.303 ms on
  // 4096 x 11008 x 4096 in either weight layout against 0.310-0.315 ms ([N][K]) and 0.338-0.346 ms ([K][N]) for the
  // 32x32x16 form; through registers 0.320-0.328 ms for [K][N] (also 4-8 % ahead on 4096^3, 8192^3 and
  // 2048 x 8192 x 2048) and level with the other form for [N][K].
  const bool m16 = s.get("M16", m16Fits && d2lFits && !clamp && bm == 256 && bn == 256 && waves == 8 && s.get("D2L", 1)) != 0;
  s.p["M16"] = m16;
  // row-major weights in other tiles than 256 columns of eight wavefronts: on request, and in the forms chosen above
  const bool d2l = m16 && s.get("D2L", d2lFits && (s.get("TB", 0) || (bn == 256 && waves == 8))) != 0;
  // a K that is no multiple of BK: the last k-tile is moved back as well, where the direct loads are used
  const bool kTail = k % bk != 0 && canShift && d2l && d2lFits;
  const bool shift = ragged && canShift && (k % bk == 0 || kTail) && (!clamp || (d2l && d2lFits));
  const bool edge = ragged && !shift;
  s.p["SHIFT"] = shift;
  if (m16 && (!m16Fits || edge)) { err = "gemm_bf16: M16 needs full 64-deep tiles, TA = 0, one staging set and no tail split"; return false; }
  s.p["D2L"] = d2l;
  if (fewRows && !(shift && clamp && d2l)) { err = "gemm_bf16: tiles of 32 rows need aligned operands and direct loads"; return false; }
  if (d2l && !d2lFits) { err = "gemm_bf16: D2L needs M16 and whole 1 KiB blocks per wavefront (row-major weights: BN = 64, 128, 192 or 256)"; return false; }
  const int64_t nbuf = s.get("NBUF", 2);
  if (nbuf < 2 || nbuf > 6 || (nbuf > 2 && (!d2l || (nbuf - 1) * (bm / 8 + bn / 8) / waves > 63))) {
    err = "gemm_bf16: NBUF is 2 to 6, more than two with direct loads only";
    return false;
  }
  s.p["NBUF"] = nbuf;
  // the 16x16x32 form's transposing reads take eight consecutive k rows of 32 bytes together: the pitch must be an odd
  // multiple of 32 bytes (through registers; direct loads leave the rows unpadded and swizzle them instead)
  if (m16 && !s.has("BPAD")) bpad = 32;
  if (d2l) bpad = 0;
  const int64_t rowA = m16 ? bk * 2 : bk * 2 + 16;
  const int64_t ldsB = s.get("TB", 0) ? bn * rowA : bk * (bn * 2 + bpad);
  const int64_t lds = nbuf * (bm * rowA + ldsB);
  if (lds > 160 * 1024) { err = "gemm_bf16: tile needs more than 160 KiB of LDS"; return false; }
  const bool outBf16 = s.get("OUT_BF16", 0) != 0;
  // staging register sets = tiles in flight from global memory; two only fit small wave tiles
  const int64_t stages = s.get("STAGES", 1);
  if (stages != 1 && stages != 2) { err = "gemm_bf16: STAGES must be 1 or 2"; return false; }
  const bool fp8 = s.get("FP8_PAIRS", 0) != 0;             // from emitGemmFp8: K counts pairs of bytes
  if (fp8 && (!d2l || edge || !s.get("TB", 0))) { err = "gemm_bf16: fp8 operands need the direct loads"; return false; }
  s.p["BM"] = bm; s.p["BN"] = bn; s.p["BK"] = bk; s.p["WM"] = wm; s.p["WN"] = wn; s.p["GROUP_M"] = gm;
  s.p["STAGES"] = stages;
  // with one wavefront per SIMD the memory instructions have to be interleaved with the MFMAs explicitly
  const bool interleave = s.get("INTERLEAVE", wm * wn <= 4) != 0;
  s.p["INTERLEAVE"] = interleave;
  const int64_t tiles = ceilDiv(m, bm) * ceilDiv(n, bn);
  int64_t skFull = 0, skUnits = 0;
  if (stages != 1 || k % bk) s.p["SK_UNITS"] = s.has("SK_UNITS") && s.get("SK_UNITS", 0) ? -1 : 0;   // needs whole k-tiles, one staging set
  if (s.get("SK_UNITS", 0) < 0) { err = "gemm_bf16: tail split needs K a multiple of BK and STAGES = 1"; return false; }
  if (!chooseTailSplit(s, tiles, ceilDiv(k, bk), batch, skFull, skUnits, err)) return false;
  s.p["SK_UNITS"] = skUnits; s.p["SK_FULL"] = skFull;

  Defines d;
  d.add("GB_NAME", s.name);
  d.add("GB_M", m); d.add("GB_N", n); d.add("GB_K", k); d.add("GB_BATCH", batch);
  d.add("GB_TA", s.get("TA", 0) ? 1 : 0); d.add("GB_TB", s.get("TB", 0) ? 1 : 0);
  d.add("GB_BM", bm); d.add("GB_BN", bn); d.add("GB_BK", bk);
  d.add("GB_WM", wm); d.add("GB_WN", wn); d.add("GB_GROUP_M", gm);
  d.add("GB_EDGE", edge ? 1 : 0);
  d.add("GB_OUT_BF16", outBf16 ? 1 : 0);
  d.add("GB_RELU", s.get("RELU", 0) ? 1 : 0);
  d.add("GB_STAGES", stages);
  d.add("GB_INTERLEAVE", interleave ? 1 : 0);
  d.add("GB_F16", s.get("F16", 0) ? 1 : 0);
  d.add("GB_BPAD", bpad);
  if (m16) d.add("GB_M16", 1);
  if (d2l) d.add("GB_D2L", 1);
  if (m16 && s.has("M16_DEAL")) d.add("GB_M16_DEAL", s.get("M16_DEAL", 0) ? 1 : 0);
  // 16-bit results of whole 256 x 256 tiles in the 16x16x32 form leave through LDS as whole rows (see the kernel)
  const bool stageOk = m16 && (bm == 256 || bm == 192) && (bn == 256 || bn == 192) && wm * wn == 8 && bm / wm / 16 % 2 == 0 && (d2l || (bm == 256 && bn == 256 && wm == 4)) && !edge &&
                       skUnits == 0 && n % 8 == 0;
  const int64_t stageC = stageOk ? std::max<int64_t>(0, std::min<int64_t>(2, s.get("STAGE_C", outBf16 ? 2 : 0))) : 0;
  s.p["STAGE_C"] = stageC;
  if (stageC) d.add("GB_STAGE_C", stageC);
  if (shift) d.add("GB_SHIFT", 1);
  if (fp8) d.add("GB_FP8", 1);
  if (nbuf > 2) d.add("GB_NBUF", nbuf);
  if (shift && clamp) d.add("GB_CLAMP", 1);
  if (kTail) d.add("GB_KTAIL", 1);
  if (s.has("BTR") && !s.get("TB", 0)) d.add("GB_BTR", s.get("BTR", 1) ? 1 : 0);
  // start of the walk along k staggered between the XCDs: default on for two k-contiguous operands (see the kernel)
  if (s.has("KROT")) d.add("GB_KROT_ON", s.get("KROT", 0) ? 1 : 0);
  if (s.get("SETPRIO", 0) > 0) d.add("GB_SETPRIO", std::min<int64_t>(3, s.get("SETPRIO", 0)));
  if (s.get("STAGGER", 0) > 0) d.add("GB_STAGGER", s.get("STAGGER", 0));
  d.add("GB_SK_UNITS", skUnits);
  d.add("GB_SK_FULL", skFull);
  src = d.wrap(kTpl_gemm_bf16);

  info.name = s.name;
  info.grid[0] = (uint32_t)(skUnits > 0 ? skFull + skUnits : tiles);
  info.grid[1] = (uint32_t)batch;
  info.block[0] = (uint32_t)(64 * wm * wn);
  info.numArgs = fp8 ? 5 : skUnits > 0 ? 4 : 3;
  info.numScalars = fp8 ? 2 : 0;
  if (skUnits > 0) {
    info.workspaceBytes = 4096 + skUnits * 2 * bm * bn * 4;
    info.workspaceArg = 3;
  }
  info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
  info.bytes = (double)batch * (2.0 * ((double)m * k + (double)k * n) + (outBf16 ? 2.0 : 4.0) * (double)m * n);
  return true;
}

bool emitGemmFp8(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  int64_t m, n, k, batch;
  if (!gemmCommon(s, err, m, n, k, batch)) return false;
  if (s.get("WAVEK", 0) > 0) return emitGemmWavek(s, src, info, err, 3, wavekAsked(s, 3), m, n, k, batch);
  const bool ta = s.get("TA", 0) != 0, tb = s.get("TB", 0) != 0;
  // As for 16 bits: where the operands' addresses are known to be aligned and no tile or switch is asked for, one of the
  // forms with direct loads, priced as a 16-bit product of half the depth.  256 x 256 tiles run on gemm_fp8_d2l.hip
  // (twice the MFMA rate), smaller ones of two k-contiguous operands on the 16-bit kernel's ring of LDS buffers (us, against
  // guarded loads: 300 x 4096 x 4096 13.9 and 17.0, 16 x 11008 x 4096 9.8 and 16.7, 700 x 2048 x 1040 7.5 and 10.5).  Whole
  // tiles of the sizes below stay with gemm_fp8.hip: its unguarded loads on the faster MFMA are ahead of the ring
  // (2048^3 12.4 against 14.6, 512 x 4096 x 4096 14.6 against 16.2; behind it only at M 64-256, K 4096, by 8-10 %).
  bool own = false;
  for (const char* key : {"BM", "BN", "BK", "WM", "WN", "D2L", "BTR", "STAGES", "PREFETCH", "ROTATE", "PINGPONG", "PERSIST", "STAGE_C", "NT_STORE", "STAGGER"}) own = own || s.has(key);
  bool shift256 = false;
  int64_t dm, dn;
  defaultGemmTile(m, n, batch, dm, dn);
  const bool whole = m % dm == 0 && n % dn == 0 && k % 128 == 0;
  if (!own && s.get("ALIGN", 0) >= 16 && shortRows(n, k) && !ta && k % 16 == 0 && n % 16 == 0 && s.get("SCALE_PTR", 0) == 0) {
    double cost;
    const Gemm16Form* tiled = chooseGemm16Form(m, n, k / 2, batch, &cost);
    WavekForm split;
    if (namesOnlyProduct(s) && wavekAhead(s, 3, tiled, cost, m, n, k, batch, split)) return emitGemmWavek(s, src, info, err, 3, split, m, n, k, batch);
  }
  if (!own && !whole && s.get("ALIGN", 0) >= 16 && shortRows(n, k) && !ta && k % 16 == 0 && n % 16 == 0 && s.get("SCALE_PTR", 0) == 0) {
    const Gemm16Form* form = chooseGemm16Form(m, n, k / 2, batch);
    // Shallow products of two k-contiguous operands lose little to guarded loads, and those run on gemm_fp8.hip's larger MFMA:
    // ahead where the choice would be 128 x 128 tiles, or 256 x 256 ones on under three quarters of the CUs (us, these and
    // guarded 128 x 128 tiles: 2000 x 5504 x 512 16.1 and 13.3, 1000 x 11008 x 1024 21.0 and 18.7, 2000 x 2816 x 1024 13.9 and 12.3;
    // x 2048 21.9 and 22.4, 2447 x 5504 x 1024 22.1 and 24.8 on 220 CUs, 700 x 5504 x 512 8.5 and 9.3 in 64 x 128)
    const bool shallow = tb && k <= 1024 && k % 128 == 0 && dm == 128 && dn == 128;
    if (form && shallow && (form->bm == 128 || (form->bm == 256 && (double)ceilDiv(m, 256) * (double)ceilDiv(n, 256) * (double)batch < 192.0))) form = nullptr;
    if (form && form->bm == 256) {
      shift256 = true;
    } else if (form && tb) {
      s.p["K"] = k / 2;
      s.p["FP8_PAIRS"] = 1;
      const bool ok = emitGemmBf16(s, src, info, err);
      s.p["K"] = k;
      s.p.erase("FP8_PAIRS");
      info.flops *= 2.0;      // two products per pair; the bytes are those of 16-bit values half as many
      return ok;
    }
  }
  if (shift256) dm = dn = 256;
  // Tiles of 192 columns where they make less of the last round idle: rounds and the part of them in use, in us at K = 4096, fitted to
  // 81 products (us, 256 and 192 columns: 2000 x 11008 x 4096 99 and 89, 1500 x 11008 x 4096 94 and 77, 3000 x 11008 x 4096 147 and 129,
  // 1500 x 4096 x 4096 row-major 53 and 41; but 4096 x 11008 x 4096 162 and 167, 2407 x 5440 x 2048 34 and 46): 23 of the 29 products
  // on 256 x 256 tiles gain 11 % on average, none loses more than 2 %.  Products of fewer than 192 columns take them too, on the guarded
  // kernel (gemm_fp8.hip), which computes less past the edge with them: row-major, us, 256 and 192 columns, 131072 x 128 x 4096 590 and
  // 167, 65536 x 176 x 512 20.8 and 18.0, 256 times 256 x 128 x 512 20.3 and 18.0, 65536 x 16 x 512 12.0 and 10.5, 512 x 176 x 1024 the same.
  if (!own && dm == 256 && dn == 256 && s.get("ALIGN", 0) >= 16 && shortRows(n, k) && !ta && n % 16 == 0 && k % 128 == 0 && m >= 256 && s.get("SCALE_PTR", 0) == 0 &&
      (shift256 || k <= 4096)) {
    auto time = [&](int64_t cols, double a, double b) {
      const double tiles = (double)ceilDiv(m, 256) * (double)ceilDiv(n, cols) * (double)batch / 256.0;
      return 2.5 + (double)k / 4096.0 * (std::ceil(tiles) * a + tiles * b);
    };
    if (time(192, 41.3, 5.8) < time(256, 47.6, 11.1)) dn = 192;
  }
  int64_t bm = s.get("BM", dm);
  int64_t bn = s.get("BN", dn);
  int64_t bk = s.get("BK", 128);
  // eight wavefronts from 128x128 up (2048^3: 1180 against 980 TFLOP/s with four)
  int64_t wm = s.get("WM", bm >= 128 && bn >= 128 ? 4 : 2), wn = s.get("WN", 2), gm = s.get("GROUP_M", 8);
  if (!checkTile(s, bm, bn, bk, wm, wn, 64, err)) return false;
  // Full 256 x 256 x 128 tiles of two k-contiguous operands: the kernel on v_mfma_f32_16x16x128 with direct loads into
  // LDS (kernels/gemm_fp8_d2l.hip), unless one of the other kernel's switches is asked for
  // Measured against the other kernel (M 4096-8192, N 4096-14336): 7-20 % faster for K up to 4096
  // (4096 x 11008 x 4096: 0.151 against 0.173 ms); beyond that level to 5 % faster on launches of more than one round
  // of tiles (8192^3: 0.419 against 0.441 ms) and 1-4 % slower on single rounds, which stay with the other.  Launches of more
  // than one round of tiles get the non-temporal result stores and the staggered start, which only pay together (see
  // the kernel); a single round is fastest without either.
  const bool legacyKnob = s.has("PREFETCH") || s.has("ROTATE") || s.has("PINGPONG") || s.has("STAGES") || (s.has("BTR") && !s.get("BTR", 1));
  const bool oneRound = ceilDiv(m, 256) * ceilDiv(n, 256) * batch <= 256;
  // (tiles of 192 columns, asked for or chosen above: moved back where they are ragged, so aligned operands are needed)
  const bool thirds = bm == 256 && bn == 192 && bk == 128 && wm == 4 && wn == 2 && m >= 256 && n >= 192 && (m % 256 == 0 || s.get("ALIGN", 0) >= 16) && (n % 192 == 0 || s.get("ALIGN", 0) >= 16) &&
                      shortRows(n, k) && s.get("PERSIST", 0) == 0 && s.get("STAGE_C", 1) != 0;
  if (s.get("D2L", !legacyKnob && (k <= 4096 || !oneRound || shift256)) && !ta && (tb || s.get("BTR", 1)) && n % 16 == 0 && bm == 256 && (bn == 256 || thirds) && bk == 128 && wm == 4 && wn == 2 &&
      (thirds || (m % 256 == 0 && n % 256 == 0) || shift256) && k % 128 == 0) {
    const int64_t scalePtr = s.get("SCALE_PTR", 0);
    if (scalePtr < 0 || scalePtr > 2) { err = "gemm_fp8: SCALE_PTR is 0 (scalar arguments), 1 (A, B, C, pointers) or 2 (A, B, pointers, C)"; return false; }
    const bool outBf16 = s.get("OUT_BF16", 0) != 0;
    // Strips of tile rows: workgroup ids are renumbered so that each of the 8 XCDs works through one contiguous run of
    // tiles; when such a run is a whole number of tile rows (at most four), the strip is the run, and all XCDs walk the
    // same columns of B at the same time (4096 x 11008 x 4096, two rows: 0.160 against 0.168 ms with strips of eight,
    // 0.164 with four); four rows otherwise (level with or ahead of eight on every shape measured).
    if (!s.has("GROUP_M")) {
      const int64_t tm = ceilDiv(m, 256), tn = ceilDiv(n, bn), run = tm * tn / 8;
      gm = (tm * tn) % 8 == 0 && run % tn == 0 && run / tn >= 1 && run / tn <= 4 ? run / tn : 4;
    }
    s.p["TA"] = 0; s.p["TB"] = tb; s.p["D2L"] = 1; s.p["BTR"] = !tb;
    s.p["BM"] = bm; s.p["BN"] = bn; s.p["BK"] = bk; s.p["WM"] = wm; s.p["WN"] = wn; s.p["GROUP_M"] = gm;
    Defines d;
    d.add("G8_NAME", s.name);
    d.add("G8_M", m); d.add("G8_N", n); d.add("G8_K", k); d.add("G8_BATCH", batch);
    d.add("G8_GROUP_M", gm);
    d.add("G8_OUT_BF16", outBf16 ? 1 : 0);
    d.add("G8_RELU", s.get("RELU", 0) ? 1 : 0);
    d.add("G8_SCALE_PTR", scalePtr);
    d.add("G8_BTR", tb ? 0 : 1);
    const int64_t tilesAll = ceilDiv(m, 256) * ceilDiv(n, bn);
    const bool moved = m % 256 || n % bn;
    if (bn != 256) d.add("G8_BN", bn);
    if (moved) d.add("G8_SHIFT", 1);
    const bool persist = s.get("PERSIST", 0) != 0 && !moved && batch == 1 && (k / 128) % 2 == 0 && tilesAll > 256;
    s.p["PERSIST"] = persist;
    if (persist) d.add("G8_PERSIST", 1);
    const bool rounds = tilesAll * batch > 256;                   // more than one round of tiles
    // The results go through LDS and leave as whole rows of the tile (STAGE_C) unless the workgroups are persistent:
    // 4096 x 11008 x 4096 0.151 against 0.160 ms, 2 to 8 % on other shapes of more than one round, level on single
    // rounds.  The staggered start then does best at half its former width.  A bf16 result, of which a lane would
    // otherwise store two bytes of a row, gains most: 0.156 ms against 0.190, and against 0.171 for the other kernel.
    const int64_t stageC = s.get("STAGE_C", 1) != 0 && !persist;
    const int64_t ntStore = s.get("NT_STORE", rounds && (stageC || !outBf16) ? 1 : 0) != 0, stagger = std::max<int64_t>(0, std::min<int64_t>(16, s.get("STAGGER", rounds ? (stageC ? 1 : 2) : 0)));
    s.p["NT_STORE"] = ntStore; s.p["STAGGER"] = stagger;
    d.add("G8_NT_STORE", ntStore);
    d.add("G8_STAGGER", stagger);
    s.p["STAGE_C"] = stageC;
    d.add("G8_STAGE_C", stageC);
    src = d.wrap(kTpl_gemm_fp8_d2l);
    info.name = s.name;
    info.grid[0] = (uint32_t)(persist ? 256 : tilesAll);
    info.grid[1] = (uint32_t)batch;
    info.block[0] = 512;
    info.numArgs = 5;
    info.numScalars = scalePtr ? 0 : 2;
    info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
    info.bytes = (double)batch * ((double)m * k + (double)k * n + (outBf16 ? 2.0 : 4.0) * (double)m * n);
    return true;
  }
  if (s.get("D2L", 0) && s.has("D2L")) { err = "gemm_fp8: D2L needs full 256 x 256 x 128 tiles, TA = 0 and TB = 1"; return false; }
  s.p["D2L"] = 0;
  // a B stored [K][N] lies in LDS as it lies in memory and is transposed by the LDS reads (BTR = 0: in registers on the way in)
  const bool btr = !tb && s.get("BTR", 1) != 0;
  s.p["BTR"] = btr;
  const int64_t lds = 2 * bm * (bk + 16) + (btr ? 2 * bk * (bn + 32) : 2 * bn * (bk + 16));
  if (lds > 160 * 1024) { err = "gemm_fp8: tile needs more than 160 KiB of LDS"; return false; }
  const bool edge = (m % bm) || (n % bn) || (k % bk);
  const bool outBf16 = s.get("OUT_BF16", 0) != 0;
  const int64_t stages = s.get("STAGES", 1);
  if (stages != 1 && stages != 2) { err = "gemm_fp8: STAGES must be 1 or 2"; return false; }
  // a second fragment set costs 8 registers per 32-row fragment: only small wave tiles can afford it
  const bool prefetch = s.get("PREFETCH", (bm / wm / 32 + bn / wn / 32) <= 4) != 0;
  s.p["PREFETCH"] = prefetch;
  s.p["TA"] = ta; s.p["TB"] = tb;
  s.p["BM"] = bm; s.p["BN"] = bn; s.p["BK"] = bk; s.p["WM"] = wm; s.p["WN"] = wn; s.p["GROUP_M"] = gm;
  s.p["STAGES"] = stages;

  Defines d;
  d.add("GF_NAME", s.name);
  d.add("GF_M", m); d.add("GF_N", n); d.add("GF_K", k); d.add("GF_BATCH", batch);
  d.add("GF_TA", ta ? 1 : 0); d.add("GF_TB", tb ? 1 : 0);
  d.add("GF_BM", bm); d.add("GF_BN", bn); d.add("GF_BK", bk);
  d.add("GF_WM", wm); d.add("GF_WN", wn); d.add("GF_GROUP_M", gm);
  d.add("GF_EDGE", edge ? 1 : 0);
  d.add("GF_OUT_BF16", outBf16 ? 1 : 0);
  d.add("GF_RELU", s.get("RELU", 0) ? 1 : 0);
  d.add("GF_STAGES", stages);
  d.add("GF_PREFETCH", prefetch ? 1 : 0);
  // fragments re-read behind their last use (no second set): where there is no room for a second set and a tile has
  // at least two k-steps
  // (default: with row-major [K][N] weights, where it measured 2-4 % faster at 4096 x 11008 x 4096; no difference with
  // [N][K] weights)
  const bool rotate = !prefetch && bk >= 128 && s.get("ROTATE", btr ? 1 : 0) != 0;
  s.p["ROTATE"] = rotate;
  d.add("GF_ROTATE", rotate ? 1 : 0);
  // the two wavefronts of a SIMD half a k-tile out of step (one k-step per tile, eight wavefronts, nothing guarded)
  const bool guarded = edge || (k % 16) || (ta && m % 16) || (!tb && n % 16);
  const bool pingpong = s.get("PINGPONG", 0) != 0 && bk == 64 && wm * wn == 8 && !guarded && !prefetch && k / bk >= stages + 2;
  s.p["PINGPONG"] = pingpong;
  d.add("GF_PINGPONG", pingpong ? 1 : 0);
  // Guarded loads of whole chunks, where the caller has looked at the operands' addresses.  In tiles of up to 128 x 128 of two
  // operands that are contiguous along k, in whole k-tiles, the compiler joins a chunk's sixteen guarded bytes by itself, behind
  // one branch for the row (1000 x 5504 x 512 9.4 us, 12.4 in chunks that are loaded in any case and then selected; 5 x 1 x 496 x
  // 1024 3.7 and 4.0; but 256 x 256 tiles 2000 x 2816 x 2048 71 and 46, a partial k-tile 2447 x 2816 x 528 16.5 and 13.3).
  const bool joined = !ta && tb && bm <= 128 && bn <= 128 && k % bk == 0;
  if (edge && !joined && s.get("ALIGN", 0) >= 16 && k % 16 == 0 && (!ta || m % 16 == 0) && (tb || n % 16 == 0)) d.add("GF_WIDE", 1);
  d.add("GF_BTR", btr ? 1 : 0);
  // where the two per-tensor scales come from: trailing scalars, or one fp32 each in device memory (graph values)
  const int64_t scalePtr = s.get("SCALE_PTR", 0);
  if (scalePtr < 0 || scalePtr > 2) { err = "gemm_fp8: SCALE_PTR is 0 (scalar arguments), 1 (A, B, C, pointers) or 2 (A, B, pointers, C)"; return false; }
  d.add("GF_SCALE_PTR", scalePtr);
  if (s.get("STAGGER", 0) > 0) d.add("GF_STAGGER", s.get("STAGGER", 0));
  src = d.wrap(kTpl_gemm_fp8);

  info.name = s.name;
  info.grid[0] = (uint32_t)(ceilDiv(m, bm) * ceilDiv(n, bn));
  info.grid[1] = (uint32_t)batch;
  info.block[0] = (uint32_t)(64 * wm * wn);
  info.numArgs = 5;       // A, B, C, scale_a, scale_b
  info.numScalars = scalePtr ? 0 : 2;
  info.flops = 2.0 * (double)batch * (double)m * (double)n * (double)k;
  info.bytes = (double)batch * ((double)m * k + (double)k * n + (outBf16 ? 2.0 : 4.0) * (double)m * n);
  return true;
}

// Attention whose wavefronts split the keys (kernels/fmha_wavek.hip).  type: 0 fp32, 1 bf16, 2 IEEE half.
static int64_t fmhaWavekLds(int type, int64_t d, int64_t qb, int64_t wk) {
  const int64_t row = d * (type == 0 ? 4 : 2);
  return wk * (std::max(32 * (2 * row + 48), 32 * (d * 4 + 16)) + 32 * qb * 8);
}

// A launch takes fewer than 2^32 threads.  Wavefronts that split the keys are more of them than those that walk: 2^23 heads of 129 queries
// under the mask are 2^32.3 in workgroups of two such wavefronts and 2^31 in pairs of 256 queries.
static bool fmhaWavekLaunches(int64_t sl, double heads, int64_t qb, int64_t wk) { return (double)ceilDiv(sl, 32 * qb) * heads * (double)(64 * wk) < 4294967296.0; }

// Wavefronts per SIMD that the registers of a form leave room for (130 to 190 of them in 16 bits, 174 to 361 in fp32).
static int64_t fmhaWavekEu(int type, int64_t d, int64_t qb) { return type != 0 ? (d <= 64 && qb == 1 ? 4 : qb == 2 && d > 64 ? 1 : 2) : d <= 64 && qb == 1 ? 2 : 1; }

bool emitFmhaWavek(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err, int type, int64_t qb, int64_t wk) {
  const int64_t b = s.p["B"], h = s.p["H"], sl = s.p["S"], dh = s.p["D"];
  const int64_t es = type == 0 ? 4 : 2;
  if ((dh != 32 && dh != 64 && dh != 128) || qb < 1 || qb > 2 || wk < 1 || wk > 16 || fmhaWavekLds(type, dh, qb, wk) > 160 * 1024 ||
      (double)sl * (double)dh * (double)es >= 2147483648.0 || !fmhaWavekLaunches(sl, (double)b * (double)h, qb, wk)) {
    err = s.family + ": WAVEK needs a head dim of 32, 64 or 128, QB 1 or 2, at most 16 wavefronts whose tiles fit 160 KiB of LDS, heads below 2 GiB, and fewer than 2^32 threads";
    return false;
  }
  if (s.f.count("SCALE") && !(s.f["SCALE"] > 0.0)) { err = s.family + ": the softmax scale must be positive"; return false; }
  const bool causal = s.get("CAUSAL", 0) != 0, out16 = type != 0 && s.get("OUT_BF16", 1) != 0;
  const double scale = s.f.count("SCALE") ? s.f["SCALE"] : 1.0;
  s.p["WAVEK"] = wk; s.p["QB"] = qb; s.p["CAUSAL"] = causal;
  s.f["SCALE"] = scale;
  Defines d;
  d.add("FW_NAME", s.name);
  d.add("FW_B", b); d.add("FW_H", h); d.add("FW_S", sl); d.add("FW_D", dh);
  d.add("FW_TYPE", type);
  d.add("FW_OUT16", out16 ? 1 : 0);
  d.add("FW_QB", qb); d.add("FW_WK", wk);
  d.add("FW_EU", std::max<int64_t>(1, s.get("EU", std::max(fmhaWavekEu(type, dh, qb), wk / 4))));
  d.add("FW_CAUSAL", causal ? 1 : 0);
  // (a power of two down to 2^-126, the smallest normal number)
  const double c = scale * 1.4426950408889634;
  const int down = type == 2 || !(c < 1.0) ? 0 : std::max(-126, std::ilogb(c));
  d.add("FW_QEXP", (int64_t)down);
  d.add("FW_C", floatLiteral(std::ldexp(c, -down)));
  src = d.wrap(kTpl_fmha_wavek);
  info.name = s.name;
  info.grid[0] = (uint32_t)(ceilDiv(sl, 32 * qb) * b * h);
  info.block[0] = (uint32_t)(64 * wk);
  info.numArgs = 4;
  info.flops = 4.0 * (double)b * h * (double)sl * sl * dh * (causal ? 0.5 : 1.0);
  info.bytes = (double)b * h * sl * dh * (3.0 * es + (out16 ? 2.0 : 4.0));
  return true;
}

// Whether wavefronts that split the keys take less time than workgroups of `br` queries that walk them (`items` of them, two query
// tiles each if `paired`, `held` by a compute unit at a time), for callers who ask for it (FILL = 2; 1: tiles that fill the part); the
// form in qb, wk.  Both times are modelled, in us: a launch, then the longer of the walk of one workgroup, in 32-key tiles times rounds, and the work
// of a compute unit; for the split also the merge and the bytes out of the L2s.  Fitted to 2600 timings of 460 launches (8 to
// 256 heads, S 64 to 2048), 10 to 22 % off on average, hence the margin: the choice is then 1.2 (bf16, head dim 64), 1.27 (128), 1.6 (fp32, 64)
// and 1.47 (128) times as fast as walks alone and no more than 5 % slower on all but one of them.  us, walk and split, D 64: bf16
// heads x S 8 x 333 7.8 and 4.7, 8 x 1024 14.5 and 7.8, 32 x 512 9.3 and 7.6; but 32 x 1024 15.8 and 17.2, 128 x 512 15.5 and 18.3; fp32
// 8 x 1024 78 and 23, 32 x 512 44 and 23, 48 x 1024 133 and 113, but 128 x 512 76 and 84.
// More workgroups than the part holds at a time take up to 1.6 times what is modelled.  Of 660 drawn launches (8 to 400 heads, S 40
// to 1600) on which the split was taken, 35 % faster on average, 34 were more than 3 % slower, most of them these: at head dim 64 in
// 16 bits 19 of 58, causal, 183 x 362 18.2 and 21.5, 371 x 1126 138 and 172.  There a walk in whole rounds is priced, its last one like the
// others, and the split taken below 0.63 of it: no loser is left, and those that go gained 1 % on average (291 x 270, whose
// walk has a second round of 35 workgroups, stays: 35.5 and 21.6).  fp32, head dim 128: not where a wavefront's second tile is the
// exception (255 x 91 causal 22.9 and 30.5).
static bool fmhaWavekAhead(const KernelSpec& s, int type, int64_t br, bool paired, double items, int64_t held, int64_t& qb, int64_t& wk) {
  const int64_t sl = s.get("S", 0), dh = s.get("D", 0);
  const double heads = (double)s.get("B", 0) * (double)s.get("H", 0);
  if (s.get("FILL", 0) < 2 || !namesOnly(s, {"B", "H", "S", "D", "CAUSAL", "OUT_BF16", "F16", "FILL"}) || (dh != 64 && dh != 128) || (double)sl * (double)dh * 4.0 >= 2147483648.0) return false;
  struct Rates { double fixed, walk, work, merge, l2, tiled, tiledWalk, tiledWork, ragged, margin; };
  static const Rates rates[2][2] = {      // 16 bits, fp32; head dim 64, 128
      {{1.94, 0.745, 0.415, 3.71, 0.0186, 2.90, 0.449, 0.104, 0.097, 0.85}, {1.87, 1.01, 0.714, 8.07, 0.0436, 3.93, 0.837, 0.179, 0.091, 0.78}},
      {{0.89, 3.07, 2.25, 8.94, 0.0007, 2.66, 2.61, 0.664, 0.017, 0.8}, {0.88, 4.94, 0.449, 18.3, 0.115, 5.70, 4.24, 1.32, 0.017, 0.78}}};
  const Rates& r = rates[type == 0][dh == 128];
  const bool causal = s.get("CAUSAL", 0) != 0;
  const double tiles = (double)ceilDiv(sl, 32), mean = causal ? (tiles + 1.0) / 2.0 : tiles;
  auto longer = [](double a, double b, double c) { return std::pow(a * a * a * a + b * b * b * b + c * c * c * c, 0.25); };
  const double each = paired ? tiles + br / 32 : causal ? (tiles + br / 32) / 2.0 : tiles;
  const double rounds = std::ceil(items / (256.0 * (double)held)), longest = causal && !paired ? tiles : each;
  const bool ragged = sl % br != 0 || sl % 64 != 0;
  const double walk = r.tiled + (1.0 + (ragged ? r.ragged : 0.0)) * longer(r.tiledWalk * rounds * longest, r.tiledWork * each * items / 256.0 * (br / 32), 0.0);
  const double busy = paired || !causal ? std::ceil(items / 256.0) : items / 256.0;
  const double whole = r.tiled + (1.0 + (ragged ? r.ragged : 0.0)) * longer(r.tiledWalk * rounds * longest, r.tiledWork * each * busy * (br / 32), 0.0);
  double least = 0.0, most = r.margin * walk;
  const int64_t row = dh * (type == 0 ? 4 : 2);
  for (int64_t q : {1, 2})
    for (int64_t w : {2, 4, 8}) {
      if ((double)w > tiles || (q == 2 && (dh == 128 || (type == 0 && w != 4))) || fmhaWavekLds(type, dh, q, w) > 160 * 1024 || !fmhaWavekLaunches(sl, heads, q, w)) continue;
      const double groups = (double)ceilDiv(sl, 32 * q) * heads, per = std::ceil(groups / 256.0);
      const int64_t fit = std::max<int64_t>(1, std::min<int64_t>(160 * 1024 / fmhaWavekLds(type, dh, q, w), fmhaWavekEu(type, dh, q) * 4 / w));
      const double turns = std::ceil(groups / (256.0 * (double)fit));
      const double chain = turns * std::ceil((turns == 1.0 ? tiles : mean) / (double)w);
      const double work = (causal ? std::max(groups / 256.0, 1.0) * 1.15 : per) * mean * (double)q / 4.0;
      const double us = r.fixed + longer(r.walk * chain, r.work * work, r.l2 * groups * mean * (double)row * 64.0 / 1e6) + r.merge * (double)(w * q) * per / 16.0;
      if (least == 0.0 || us < least) {
        least = us; qb = q; wk = w; most = r.margin * walk;
        if (turns > 1.0 && type != 0 && dh == 64) most = std::min(most, 0.63 * whole);
        if (turns > 1.0 && type == 0 && dh == 128 && tiles < 2.0 * (double)w) most = 0.0;
      }
    }
  return least > 0.0 && least < most;
}

bool emitFmhaBf16(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  if (!need(s, {"B", "H", "S", "D"}, err) || !positive(s, {"B", "H", "S", "D"}, err)) return false;
  const int64_t b = s.p["B"], h = s.p["H"], sl = s.p["S"], dh = s.p["D"];
  if (s.get("WAVEK", 0) > 0) return emitFmhaWavek(s, src, info, err, s.get("F16", 0) ? 2 : 1, s.get("QB", 1), s.get("WAVEK", 0));
  if (dh % 32 || dh > 256) { err = "fmha_bf16: head dim must be a multiple of 32, at most 256"; return false; }
  int64_t br = s.get("BR", 0), bc = s.get("BC", 0);
  // A sequence length that the tiles do not divide is taken too (the kernel guards its last query and key tiles); the
  // automatic choice prefers tiles that divide it, and for a length with no such tile takes the sizes of its magnitude.
  // Large tiles with a guarded edge are faster than small ones that divide the length: 32 queries per workgroup (one
  // wavefront) for a length like 4000 ran at a fifth of the speed of 256 with the last tile partly filled.
  if (br <= 0) {
    if (sl % 256 == 0) br = 256;
    else if (sl % 128 == 0) br = 128;
    else if (sl % 64 == 0 && sl <= 512) br = 64;
    else br = sl > 128 ? 256 : (sl > 64 ? 128 : (sl > 32 ? 64 : 32));
  }
  // Launches that leave half the compute units or more without a workgroup of 256 queries (under the mask: without a pair of
  // query tiles) take 128 queries per workgroup instead, and under the mask pairs only where enough of them are left for every
  // CU: the pairs balance the work of a full part, on an emptier one they halve its parallelism (us, before and now: B2 H16
  // S777 D64 19.4 and 15.4, causal 29.7 and 16.0; B1 H8 S2048 D64 36.0 and 25.6, causal 44.7 and 26.5; B3 H12 S1300 D64 causal
  // 38.8 and 26.9; B1 H32 S2048 D128 causal 69.3 and 57.3, with pairs).  Above that 256 stays ahead: B3 H12 S1300 D64 with 216
  // workgroups 28.5 against 31.4; causal with 192 pairs B4 H32 S600 D128 41 against 64, B4 H12 S2048 D64 46 against 61.
  const bool masked = s.get("CAUSAL", 0) != 0;
  bool own = !s.get("FILL", 0) || s.get("BR", 0) > 0 || s.get("BC", 0) > 0 || s.get("QW", 0) > 0;    // (on request: FILL)
  for (const char* key : {"D2L", "PAIR", "PERSIST", "OCC", "STAGE_O"}) own = own || s.has(key);
  const double heads = (double)b * (double)h, jobs = (double)ceilDiv(sl, br) * heads / (masked && ((b * h) % 2 == 0 || ceilDiv(sl, br) % 2 == 0) ? 2.0 : 1.0);
  bool noPair = false;
  // Under the mask at head dims above 96, whose workgroups have a CU to themselves, more than 256 of 128 queries are a second round
  // while those of 256 by themselves are still one: heads x S, D 128, us, pairs of 256, 128 and 256 by themselves, 60 x 1024 46.9,
  // 56.2, 37.8; 80 x 768 41.4, 44.0, 30.4; 64 x 600 40.3, 30.7, 25.2; but 16 x 2048, 256 of 128, 67.1, 46.8, 55.9.
  if (!own && jobs <= 128.0) {
    const double small = (double)ceilDiv(sl, 128) * heads;
    const bool oneRound = masked && dh > 96 && br == 256 && small > 256.0 && small < 512.0;
    if (br == 256 && !oneRound) br = 128;
    noPair = masked && (oneRound || (double)ceilDiv(sl, br) * heads / 2.0 < 256.0);
  }
  if (bc <= 0) {
    bc = sl > 32 ? 64 : 32;
    if (2 * bc * (dh * 2 + 16) + 3 * bc * (dh * 2 + 32) > 160 * 1024) bc = 32;   // head dim 256: 64-key tiles do not fit the LDS
  }
  if (br % 32 || br > 512 || bc % 32) { err = "fmha_bf16: BR must be a multiple of 32 (at most 512) and BC a multiple of 32"; return false; }
  // 64 queries per wavefront (every LDS fragment feeds two MFMAs, one wavefront per SIMD with the whole
  // register file) when that still leaves four wavefronts and the step-pipelined loop applies
  int64_t qw = s.get("QW", 0);
  if (qw <= 0) qw = 1;
  if ((qw != 1 && qw != 2) || br % (32 * qw)) { err = "fmha_bf16: QW must be 1 or 2 and BR a multiple of 32 * QW"; return false; }
  const bool ragged = sl % br != 0 || sl % bc != 0;
  if (ragged && (double)sl * (double)dh * 2.0 >= 4294967296.0) {
    err = "fmha_bf16: a sequence length that is no multiple of the tiles needs heads below 4 GiB";
    return false;
  }
  if ((double)ceilDiv(sl, br) * (double)b * (double)h > 2147483647.0) { err = "fmha_bf16: too many workgroups"; return false; }
  if (s.f.count("SCALE") && !(s.f["SCALE"] > 0.0)) { err = "fmha_bf16: the softmax scale must be positive"; return false; }
  const int64_t vpad = s.get("VPAD", 32);
  if (vpad < 0 || vpad % 16) { err = "fmha_bf16: VPAD must be a multiple of 16 bytes"; return false; }
  const int64_t lds = 2 * bc * (dh * 2 + 16) + 3 * bc * (dh * 2 + vpad);   // two K buffers, three V buffers
  if (lds > 160 * 1024) { err = "fmha_bf16: tile needs more than 160 KiB of LDS"; return false; }
  const bool causal = s.get("CAUSAL", 0) != 0, outBf16 = s.get("OUT_BF16", 1) != 0;
  const double scale = s.f.count("SCALE") ? s.f["SCALE"] : 1.0;
  if (!own) {
    const bool two = causal && !noPair && ((b * h) % 2 == 0 || ceilDiv(sl, br) % 2 == 0);
    int64_t splitQb, splitWk;
    if (fmhaWavekAhead(s, s.get("F16", 0) ? 2 : 1, br, two, (double)ceilDiv(sl, br) * heads / (two ? 2.0 : 1.0), std::max<int64_t>(1, 8 / (br / 32)), splitQb, splitWk))
      return emitFmhaWavek(s, src, info, err, s.get("F16", 0) ? 2 : 1, splitQb, splitWk);
  }
  s.p["BR"] = br; s.p["BC"] = bc; s.p["QW"] = qw; s.p["CAUSAL"] = causal; s.p["OUT_BF16"] = outBf16;
  s.f["SCALE"] = scale;

  Defines d;
  d.add("FA_NAME", s.name);
  d.add("FA_B", b); d.add("FA_H", h); d.add("FA_S", sl); d.add("FA_D", dh);
  d.add("FA_BR", br); d.add("FA_BC", bc); d.add("FA_QW", qw);
  d.add("FA_CAUSAL", causal ? 1 : 0);
  d.add("FA_C", floatLiteral(scale * 1.4426950408889634));
  d.add("FA_OUT_BF16", outBf16 ? 1 : 0);
  d.add("FA_F16", s.get("F16", 0) ? 1 : 0);
  d.add("FA_VPAD", vpad);
  // K and V tiles straight from global memory into LDS (see the kernel): head dim 128, 64-key tiles, eight wavefronts of
  // 32 queries, whole tiles.  On request for now.
  const bool d2lFits = dh == 128 && bc == 64 && br == 256 && qw == 1 && !ragged;
  const bool d2l = s.get("D2L", 0) != 0;
  if (d2l && !d2lFits) { err = "fmha_bf16: D2L needs head dim 128, BC = 64, BR = 256, QW = 1 and a sequence length that is a multiple of 256"; return false; }
  s.p["D2L"] = d2l;
  if (d2l) d.add("FA_D2L", 1);
  // causal: a workgroup takes a pair of query tiles with the same total number of key tiles, unless asked not to:
  // PAIR = 1 of one head (an even number of query tiles), PAIR = 2 of two heads (an even number of heads; see the kernel)
  // (across two heads by default: the same speed as within one head, 641 against 763 MB of HBM traffic at B8 H32 S2048 D128)
  int64_t pairMode = causal ? s.get("PAIR", noPair ? 0 : (b * h) % 2 == 0 ? 2 : 1) : 0;
  if (pairMode == 2 && (b * h) % 2) pairMode = 1;
  if (pairMode == 1 && ceilDiv(sl, br) % 2) pairMode = 0;
  if (pairMode < 0 || pairMode > 2) { err = "fmha_bf16: PAIR is 0, 1 or 2"; return false; }
  const bool pair = pairMode != 0;
  s.p["PAIR"] = pairMode;
  d.add("FA_PAIR", pairMode);
  // One workgroup per compute unit that works through its query tiles one after the other and fetches the next one's
  // first tiles while it finishes the current one, where every job has the same length (no mask, or pairs) and an even
  // number of key tiles (the fetch sits in the iteration known at compile time to be the last).
  const int64_t nq = ceilDiv(sl, br), items = (pairMode == 2 ? nq * (b * h / 2) : (pair ? nq / 2 : nq) * b * h);
  const bool even = !ragged && (causal ? br % (2 * bc) == 0 : (sl / bc) % 2 == 0);
  // Only where the steady-state form of the iteration exists (64-key tiles, head dim a multiple of 64): measured with the
  // general form alone (head dim 96, 256) the persistent kernel is up to 1.8 times slower than one job per workgroup.
  const bool steady = bc == 64 && dh % 64 == 0 && qw == 1;
  const bool persist = s.get("PERSIST", steady ? 1 : 0) != 0 && (!causal || pair) && even && items > 256;
  s.p["PERSIST"] = persist;
  d.add("FA_PERSIST", persist ? 1 : 0);
  // The result tile goes through LDS to be written in whole rows, where that was measured to pay: not for the pairs of
  // query tiles under a causal mask unless the workgroup is persistent (the second pass runs while the first one's
  // scattered stores drain, and the detour costs time).
  if (s.get("STAGE_O", causal && !persist ? 0 : 1) == 0) d.add("FA_STAGE_O", "0");
  // two wavefronts per SIMD: one workgroup of 8 wavefronts, or two smaller ones when the LDS holds both
  int64_t occ = s.get("OCC", 0);
  if (occ <= 0) occ = (br >= 256 || qw == 2 || 2 * lds > 160 * 1024) ? 1 : 2;
  s.p["OCC"] = occ;
  d.add("FA_OCC", occ);
  src = d.wrap(kTpl_fmha_bf16);

  info.name = s.name;
  info.grid[0] = (uint32_t)(persist ? 256 : items);      // persistent: the compute units of an MI355X
  info.block[0] = (uint32_t)(2 * br / qw);
  info.numArgs = 4;
  // two products of S x S x D per head; a causal mask leaves half of each
  info.flops = 4.0 * (double)b * h * (double)sl * sl * dh * (causal ? 0.5 : 1.0);
  info.bytes = (double)b * h * sl * dh * (3 * 2.0 + (outBf16 ? 2.0 : 4.0));
  return true;
}

bool emitFmhaF32(KernelSpec& s, std::string& src, KernelLaunchInfo& info, std::string& err) {
  if (!need(s, {"B", "H", "S", "D"}, err) || !positive(s, {"B", "H", "S", "D"}, err)) return false;
  const int64_t b = s.p["B"], h = s.p["H"], sl = s.p["S"], dh = s.p["D"];
  if (s.get("WAVEK", 0) > 0) return emitFmhaWavek(s, src, info, err, 0, s.get("QB", 1), s.get("WAVEK", 0));
  if (dh % 32 || dh > 256) { err = "fmha_f32: head dim must be a multiple of 32, at most 256"; return false; }
  bool own = false;
  for (const char* key : {"BR", "BC", "D2L", "OCC", "PAIR"}) own = own || s.has(key);
  // queries per workgroup (32 per wavefront): four wavefronts, fewer for short sequences
  int64_t br = s.get("BR", 0);
  bool halved = false;
  if (br <= 0) {
    br = sl >= 128 ? 128 : (sl > 64 ? 128 : (sl > 32 ? 64 : 32));
    // Under the mask at head dims above 64, a launch of 256 to 512 workgroups is one round that lasts as long as the longest query
    // tile of a head.  Tiles of half the size in pairs, the longest with the shortest, all last the same (heads x S, D 128, us
    // with tiles of 128, of 64 by themselves and in pairs: 112 x 512 138, 168, 102; 32 x 2048 520, -, 340; 90 x 384 89, 89, 80).  An
    // odd number of them has no pairs and gains while they fill the part once and two thirds (80 x 448 123, 78; 40 x 1344 346, 287;
    // 100 x 576 152, 162); a last tile partly filled loses (80 x 600 134, 205).  One round of 128 or less loses, B1 H32 S1024 D128
    // 146 and 166, more gain nothing, B8 H32 S640 D128 342 and 350.
    const double tiles = (double)ceilDiv(sl, 128) * (double)b * (double)h;
    if (s.get("FILL", 0) && s.get("CAUSAL", 0) && dh > 64 && br == 128 && !s.has("PAIR") && !s.has("D2L") && tiles > 256.0 && tiles <= 512.0 && sl % 64 == 0 &&
        (sl % 128 == 0 || (double)(sl / 64) * (double)b * (double)h <= 853.0)) {
      br = 64;
      halved = sl % 128 == 0;
    }
  }
  if (br % 32 || br > 512) { err = "fmha_f32: BR must be a multiple of 32, at most 512"; return false; }
  // keys per LDS tile: 64 for head dims above 64 while two workgroups' tiles fit the LDS together, else 32 (measured at
  // B8 H32 S2048: head dim 64 135 against 131 TFLOP/s with 32-key tiles, head dim 128 the same either way)
  int64_t bc = s.get("BC", 0);
  // whole tiles of head dim 64 or 128 can have their K and V tiles straight from global memory into two LDS buffers each
  // (see the kernel): the default at head dim 128 (B8 H32 S2048 causal: 2.70 against 2.80 ms); at head dim 64, where a
  // workgroup's loads are short next to its MFMAs, the two workgroups of a CU hide them as well (2.06 against 2.02 ms)
  const bool d2lShape = (dh == 64 || dh == 128) && sl % br == 0;
  bool d2l = s.get("D2L", dh == 128 ? 1 : 0) != 0 && d2lShape;
  auto ldsOf = [&](int64_t keys) { return d2l ? 4 * keys * dh * 4 : keys * ((dh + 4) + (dh + 8)) * 4; };
  if (bc <= 0) bc = (sl > 32 && dh > 64 && 2 * ldsOf(64) <= 160 * 1024) ? 64 : 32;
  if (bc % 32 || bc <= 0) { err = "fmha_f32: BC must be a multiple of 32"; return false; }
  if (d2l && sl % bc) d2l = false;
  if (ldsOf(bc) > 160 * 1024) { err = "fmha_f32: the key tile needs more than 160 KiB of LDS"; return false; }
  if ((double)ceilDiv(sl, br) * (double)b * (double)h > 2147483647.0) { err = "fmha_f32: too many workgroups"; return false; }
  if ((double)sl * (double)dh >= 2147483648.0) { err = "fmha_f32: a head must have fewer than 2^31 elements"; return false; }
  if (s.f.count("SCALE") && !(s.f["SCALE"] > 0.0)) { err = "fmha_f32: the softmax scale must be positive"; return false; }
  const bool causal = s.get("CAUSAL", 0) != 0;
  const double scale = s.f.count("SCALE") ? s.f["SCALE"] : 1.0;
  // registers: Q fragments and the output accumulators take D / 2 each; beyond D = 128 a wavefront needs the whole file
  int64_t occ = s.get("OCC", 0);
  if (occ <= 0) occ = (dh > 128 || 2 * ldsOf(bc) > 160 * 1024) ? 1 : 2;
  // under the mask a workgroup may take two query tiles of its head, the longest with the shortest (see the kernel)
  const int64_t nq = ceilDiv(sl, br);
  const bool pairFits = causal && nq % 2 == 0;
  // the default once the halved grid still gives every CU its two workgroups (B8 H32 S2048 causal: head dim 128 2.19
  // against 2.70 ms, head dim 64 1.18 against 1.45 ms; on grids smaller than the part it costs parallelism: 20 workgroups
  // instead of 40 at B1 H5 S1024 take 0.129 against 0.114 ms)
  const bool pair = s.get("PAIR", pairFits && (halved || (nq / 2) * b * h >= 512) ? 1 : 0) != 0;
  if (pair && !pairFits) { err = "fmha_f32: PAIR needs the causal mask and an even number of query tiles"; return false; }
  // (not where the direct loads are the default: with and without them the kernel gives the same bits, which a split would not)
  if (!own && !d2l) {
    int64_t splitQb, splitWk;
    if (fmhaWavekAhead(s, 0, br, pair, (double)((pair ? nq / 2 : nq) * b * h), std::max<int64_t>(1, 4 * occ / (br / 32)), splitQb, splitWk))
      return emitFmhaWavek(s, src, info, err, 0, splitQb, splitWk);
  }
  s.p["BR"] = br; s.p["BC"] = bc; s.p["CAUSAL"] = causal; s.p["OCC"] = occ; s.p["D2L"] = d2l; s.p["PAIR"] = pair;
  s.f["SCALE"] = scale;

  Defines d;
  d.add("FF_NAME", s.name);
  d.add("FF_PAIR", pair ? 1 : 0);
  d.add("FF_B", b); d.add("FF_H", h); d.add("FF_S", sl); d.add("FF_D", dh);
  d.add("FF_WAVES", br / 32); d.add("FF_BC", bc);
  d.add("FF_CAUSAL", causal ? 1 : 0);
  d.add("FF_C", floatLiteral(scale * 1.4426950408889634));
  d.add("FF_OCC", occ);
  d.add("FF_D2L", d2l ? 1 : 0);
  src = d.wrap(kTpl_fmha_f32);

  info.name = s.name;
  info.grid[0] = (uint32_t)((pair ? nq / 2 : nq) * b * h);
  info.block[0] = (uint32_t)(2 * br);
  info.numArgs = 4;
  info.flops = 4.0 * (double)b * h * (double)sl * sl * dh * (causal ? 0.5 : 1.0);
  info.bytes = (double)b * h * sl * dh * 4 * 4.0;
  return true;
}

}  // namespace

const std::string& prelude() {
  static const std::string text(kTpl_common);
  return text;
}

bool emitKernel(KernelSpec& spec, std::string& src, KernelLaunchInfo& info, std::string& err) {
  src.clear();
  err.clear();
  info = KernelLaunchInfo();
  if (spec.name.empty()) { err = "kernel name is empty"; return false; }
  for (char c : spec.name)
    if (!(isalnum((unsigned char)c) || c == '_')) { err = "kernel name must be a C identifier"; return false; }
  if (spec.family == "layernorm") return emitLayerNorm(spec, src, info, err);
  if (spec.family == "elementwise") return emitElementwise(spec, src, info, err);
  if (spec.family == "binary") return emitBinary(spec, src, info, err);
  if (spec.family == "gather") return emitGather(spec, src, info, err);
  if (spec.family == "softmax") return emitSoftmax(spec, src, info, err);
  if (spec.family == "gemm_f32") return emitGemmF32(spec, src, info, err);
  if (spec.family == "gemm_f64") return emitGemmF64(spec, src, info, err);
  if (spec.family == "gemm_bf16") return emitGemmBf16(spec, src, info, err);
  if (spec.family == "gemm_fp8") return emitGemmFp8(spec, src, info, err);
  if (spec.family == "fmha_bf16") return emitFmhaBf16(spec, src, info, err);
  if (spec.family == "fmha_f32") return emitFmhaF32(spec, src, info, err);
  err = "unknown kernel family '" + spec.family + "'";
  return false;
}

}  // namespace hipgen
}  // namespace KernelCodeGen
