// Runtime specialisation of the streaming kernel (hipRTC).
//
// The build-time catalogue covers the common shapes over floating-point
// storage types.  A call outside it -- a user offset list (Positional,
// NamedStencil, src/stencils/positional.jl:55-62, named.jl:61-81) or an
// integer / Bool element type -- would otherwise run the runtime-offset LDS
// tile kernel, which reads its offsets from a table.  Here the library
// writes the call's shape as a compile-time offset table, compiles
// stream_kernel<S, op, shape, V, KY> for gfx950 with hipRTC from the kernel
// headers embedded in the library at build time, and loads it as a module:
// the same kernel, with the same fold expressions, that the catalogue
// shapes run.
//
// Compiled code objects are cached in the process (per device) and on disk
// (STH_JIT_CACHE, else $XDG_CACHE_HOME/stencils_hip, else
// ~/.cache/stencils_hip), keyed by a hash of the generated source, the
// embedded headers and the compile options.  A failed compile is
// remembered and the call keeps the runtime-offset kernel (a failed load is
// tried again on the next call).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <sys/stat.h>
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "common.hpp"

namespace sth {

// Generated by build.py (jit_sources.hip): the kernel headers as text and the
// device compile options of the library's own build.
extern const int kJitHeaderCount;
extern const char* const kJitHeaderNames[];
extern const char* const kJitHeaderTexts[];
extern const int kJitOptionCount;
extern const char* const kJitOptions[];

// Stand-ins for the system headers the kernel headers include: hipRTC
// declares the HIP device runtime itself and ships no C library headers.
// The host launchers in the headers are parsed but never used here.
inline const char* jit_stub_hip_runtime() {
  return "#pragma once\n"
         "typedef struct ihipStream_t* hipStream_t;\n"
         "#define hipLaunchKernelGGL(...) ((void)0)\n";
}
inline const char* jit_stub_type_traits() {
  return "#pragma once\n"
         "namespace std {\n"
         "template <class T, T v> struct integral_constant {\n"
         "  static constexpr T value = v;\n"
         "  constexpr operator T() const { return v; }\n"
         "};\n"
         "using true_type = integral_constant<bool, true>;\n"
         "using false_type = integral_constant<bool, false>;\n"
         "}  // namespace std\n";
}
inline const char* jit_stub_stdint() {
  return "#pragma once\n"
         "typedef signed char int8_t; typedef unsigned char uint8_t;\n"
         "typedef short int16_t; typedef unsigned short uint16_t;\n"
         "typedef int int32_t; typedef unsigned int uint32_t;\n"
         "typedef long int64_t; typedef unsigned long uint64_t;\n"
         "typedef long intptr_t; typedef unsigned long uintptr_t;\n";
}

// Largest reach per axis specialised at run time: a lane holds its rows plus
// the reach on either side in registers, as the catalogue's shapes do (up
// to Window(3) and Circle(3)).
constexpr int kJitMaxReach = 3;

// Whether a call of `cells` cells compiles a specialisation: the first call
// of each shape pays for one compile (about half a second, or a read of the
// disk cache), so only arrays of at least STH_JIT_MIN_CELLS cells (default
// 2^20) do; STH_JIT=0 turns the path off and STH_JIT=1 takes it for every
// size.
inline bool jit_wanted(int64_t cells) {
  static const int mode = [] {
    const char* e = std::getenv("STH_JIT");
    return e ? std::atoi(e) : -1;
  }();
  static const int64_t min_cells = [] {
    const char* e = std::getenv("STH_JIT_MIN_CELLS");
    return e ? std::atoll(e) : (int64_t(1) << 20);
  }();
  if (mode == 0) return false;
  if (mode == 1) return true;
  return cells >= min_cells;
}

// STH_JIT_VERBOSE=1: say on stderr why a call keeps the runtime-offset or
// tiled kernel (a failed compile or load).
inline void jit_note(const std::string& what, const std::string& why) {
  static const bool verbose = [] {
    const char* e = std::getenv("STH_JIT_VERBOSE");
    return e && std::atoi(e) != 0;
  }();
  if (verbose) std::fprintf(stderr, "stencils_hip: %s not specialised: %s\n", what.c_str(), why.c_str());
}

// Storage type name of an sth_dtype, as written at global scope.
inline const char* jit_type_name(int dtype) {
  switch (dtype) {
    case STH_BOOL: return "bool";
    case STH_U8: return "uint8_t";
    case STH_I8: return "int8_t";
    case STH_U16: return "uint16_t";
    case STH_I16: return "int16_t";
    case STH_U32: return "uint32_t";
    case STH_I32: return "int32_t";
    case STH_U64: return "uint64_t";
    case STH_I64: return "int64_t";
    case STH_F32: return "float";
    case STH_F64: return "double";
    case STH_BF16: return "sth::bf16_t";
    case STH_F16: return "sth::f16_t";
    default: return nullptr;
  }
}

inline uint64_t jit_fnv1a(const std::string& s, uint64_t h = 1469598103934665603ull) {
  for (unsigned char c : s) {
    h ^= c;
    h *= 1099511628211ull;
  }
  return h;
}

struct JitKernel {
  hipModule_t mod = nullptr;
  hipFunction_t fn = nullptr;
  std::string name;  // variant name shown by the tuning table
  bool failed = false;
};

inline std::mutex& jit_mutex() {
  static std::mutex m;
  return m;
}
inline std::map<std::string, JitKernel>& jit_cache() {
  static std::map<std::string, JitKernel> c;
  return c;
}

inline std::string jit_cache_dir() {
  if (const char* d = std::getenv("STH_JIT_CACHE")) return d;
  if (const char* x = std::getenv("XDG_CACHE_HOME")) return std::string(x) + "/stencils_hip";
  if (const char* h = std::getenv("HOME")) return std::string(h) + "/.cache/stencils_hip";
  return "";
}

inline bool jit_read_file(const std::string& path, std::string* out) {
  FILE* f = std::fopen(path.c_str(), "rb");
  if (!f) return false;
  std::string s;
  char buf[65536];
  size_t n;
  while ((n = std::fread(buf, 1, sizeof buf, f)) > 0) s.append(buf, n);
  std::fclose(f);
  *out = std::move(s);
  return true;
}

inline void jit_write_file(const std::string& dir, const std::string& name, const std::string& data) {
  if (dir.empty()) return;
  // mkdir -p
  for (size_t i = 1; i <= dir.size(); ++i)
    if (i == dir.size() || dir[i] == '/') mkdir(dir.substr(0, i).c_str(), 0755);
  const std::string tmp = dir + "/" + name + ".tmp" + std::to_string(getpid());
  FILE* f = std::fopen(tmp.c_str(), "wb");
  if (!f) return;
  const bool ok = std::fwrite(data.data(), 1, data.size(), f) == data.size();
  std::fclose(f);
  if (ok) std::rename(tmp.c_str(), (dir + "/" + name).c_str());
  else std::remove(tmp.c_str());
}

// Compile `src` (which instantiates the kernel named by `expr`) with hipRTC;
// returns the code object and the kernel's lowered name.
inline bool jit_compile(const std::string& src, const std::string& expr, std::string* code, std::string* lowered,
                        std::string* log) {
  std::vector<const char*> names, texts;
  for (int i = 0; i < kJitHeaderCount; ++i) {
    names.push_back(kJitHeaderNames[i]);
    texts.push_back(kJitHeaderTexts[i]);
  }
  names.push_back("hip/hip_runtime.h");
  texts.push_back(jit_stub_hip_runtime());
  names.push_back("stdint.h");
  texts.push_back(jit_stub_stdint());
  names.push_back("stddef.h");
  texts.push_back("#pragma once\n");
  names.push_back("type_traits");
  texts.push_back(jit_stub_type_traits());
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "sth_jit.hip", static_cast<int>(names.size()), texts.data(),
                          names.data()) != HIPRTC_SUCCESS) {
    *log = "hiprtcCreateProgram failed";
    return false;
  }
  hiprtcAddNameExpression(prog, expr.c_str());
  const hiprtcResult rc = hiprtcCompileProgram(prog, kJitOptionCount, const_cast<const char**>(kJitOptions));
  size_t ls = 0;
  hiprtcGetProgramLogSize(prog, &ls);
  log->assign(ls, '\0');
  if (ls) hiprtcGetProgramLog(prog, &(*log)[0]);
  bool ok = rc == HIPRTC_SUCCESS;
  if (ok) {
    const char* ln = nullptr;
    size_t cs = 0;
    ok = hiprtcGetLoweredName(prog, expr.c_str(), &ln) == HIPRTC_SUCCESS && ln &&
         hiprtcGetCodeSize(prog, &cs) == HIPRTC_SUCCESS && cs > 0;
    if (ok) {
      *lowered = ln;
      code->assign(cs, '\0');
      ok = hiprtcGetCode(prog, &(*code)[0]) == HIPRTC_SUCCESS;
    }
  }
  hiprtcDestroyProgram(&prog);
  return ok;
}

// The shape as a compile-time offset table: struct sth::jit::<name>
// (Shape unless a kernel needs several).
inline std::string jit_shape_source(int L, const int8_t* offs3, int rx, int ry, int rz,
                                    const std::string& name = "Shape") {
  std::string table;
  for (int k = 0; k < L; ++k) {
    if (k) table += ", ";
    table += "{" + std::to_string(offs3[3 * k]) + ", " + std::to_string(offs3[3 * k + 1]) + ", " +
             std::to_string(offs3[3 * k + 2]) + "}";
  }
  return "namespace sth {\nnamespace jit {\n"
         "struct " + name + " {\n"
         "  static constexpr bool kStatic = true;\n"
         "  static constexpr int L = " + std::to_string(L) + ", RX = " + std::to_string(rx) +
         ", RY = " + std::to_string(ry) + ", RZ = " + std::to_string(rz) + ";\n"
         "  static constexpr int8_t off[" + std::to_string(L) + "][3] = {" + table + "};\n"
         "};\n}  // namespace jit\n}  // namespace sth\n";
}

// Compile (or find in the caches) `src`, which instantiates the kernel
// `expr` names, and load it on the current device; nullptr when it cannot
// be built (`why` says why).  `label` names the variant.
inline const JitKernel* jit_load(const std::string& src, const std::string& expr, const std::string& label,
                                 std::string* why) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    *why = "no device";
    return nullptr;
  }
  std::lock_guard<std::mutex> lk(jit_mutex());
  JitKernel& jk = jit_cache()[std::to_string(dev) + "\n" + src];
  if (jk.fn) return &jk;
  if (jk.failed) {
    *why = "an earlier compile of this kernel failed";
    return nullptr;
  }
  // the disk cache's key covers everything that shapes the code object
  std::string all = src + expr;
  for (int i = 0; i < kJitHeaderCount; ++i) all += kJitHeaderTexts[i];
  for (int i = 0; i < kJitOptionCount; ++i) all += kJitOptions[i];
  char hex[17];
  std::snprintf(hex, sizeof hex, "%016llx", static_cast<unsigned long long>(jit_fnv1a(all)));
  const std::string dir = jit_cache_dir();
  std::string code, lowered, log;
  bool have = !dir.empty() && jit_read_file(dir + "/" + hex + ".co", &code) &&
              jit_read_file(dir + "/" + hex + ".name", &lowered) && !code.empty() && !lowered.empty();
  if (!have) {
    if (!jit_compile(src, expr, &code, &lowered, &log)) {
      jk.failed = true;
      *why = "hipRTC: " + log.substr(0, 400);
      return nullptr;
    }
    jit_write_file(dir, std::string(hex) + ".co", code);
    jit_write_file(dir, std::string(hex) + ".name", lowered);
  }
  if (hipModuleLoadData(&jk.mod, code.data()) != hipSuccess ||
      hipModuleGetFunction(&jk.fn, jk.mod, lowered.c_str()) != hipSuccess) {
    // not remembered: a load refused now (under another thread's stream
    // capture, say) may succeed on a later call; the code object is cached
    (void)hipGetLastError();
    if (jk.mod) (void)hipModuleUnload(jk.mod);
    jk.mod = nullptr;
    jk.fn = nullptr;
    *why = "module load failed";
    return nullptr;
  }
  jk.name = "jit_" + std::string(hex) + "/" + label;
  return &jk;
}

// A specialisation already loaded, by what it was asked for: the kernel's
// kind and its parameters as bytes, so that a call need not write out the
// source to look it up.  A kernel that could not be built or loaded is not
// kept here.
struct JitRequest {
  std::string key;
  explicit JitRequest(char kind) {
    int dev = -1;
    (void)hipGetDevice(&dev);
    key.push_back(kind);
    add(dev);
  }
  JitRequest& add(int v) {
    key.append(reinterpret_cast<const char*>(&v), sizeof v);
    return *this;
  }
  template <class T>
  JitRequest& add(const T* v, size_t n) {
    add(static_cast<int>(n));
    key.append(reinterpret_cast<const char*>(v), n * sizeof(T));
    return *this;
  }
};
template <class Build>
inline const JitKernel* jit_remembered(const JitRequest& r, Build&& build) {
  static std::mutex m;
  static std::map<std::string, const JitKernel*> known;
  {
    std::lock_guard<std::mutex> lk(m);
    const auto it = known.find(r.key);
    if (it != known.end()) return it->second;
  }
  const JitKernel* k = build();
  if (k) {
    std::lock_guard<std::mutex> lk(m);
    known.emplace(r.key, k);
  }
  return k;
}

// The source of the streaming kernel specialised to one shape (L offsets, x
// fastest, as int8 triples) for storage type `dtype`, fold `opk`, V cells per
// lane and KY rows per lane (false: no type name).
inline bool jit_stream_source(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int rz, int v, int ky,
                              std::string* src_out, std::string* expr_out) {
  const char* tn = jit_type_name(dtype);
  if (!tn) return false;
  const std::string targs = std::string(tn) + ", " + std::to_string(opk) + ", sth::jit::Shape, " +
                            std::to_string(v) + ", " + std::to_string(ky);
  *src_out = "#include \"stream_kernel.hpp\"\n" + jit_shape_source(L, offs3, rx, ry, rz) +
             "namespace sth {\ntemplate __global__ void stream_kernel<" + targs + ">(MapParams);\n}  // namespace sth\n";
  *expr_out = "&sth::stream_kernel<" + targs + ">";
  return true;
}

// It, loaded on the current device.
inline const JitKernel* jit_stream_kernel(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int rz,
                                          int v, int ky, std::string* why) {
  const JitRequest request = JitRequest('s').add(dtype).add(opk).add(rx).add(ry).add(rz).add(v).add(ky).add(offs3, 3 * static_cast<size_t>(L));
  return jit_remembered(request, [&]() -> const JitKernel* {
    std::string src, expr;
    if (!jit_stream_source(dtype, opk, L, offs3, rx, ry, rz, v, ky, &src, &expr)) {
      *why = "no type name";
      return nullptr;
    }
    return jit_load(src, expr, "stream" + std::to_string(v) + "x" + std::to_string(ky), why);
  });
}

// The one-byte extremes kernel (bytes_kernel) specialised to one shape.
inline bool jit_bytes_source(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int ky,
                             std::string* src_out, std::string* expr_out) {
  const char* tn = jit_type_name(dtype);
  if (!tn) return false;
  const std::string targs = std::string(tn) + ", " + std::to_string(opk) + ", sth::jit::Shape, " + std::to_string(ky);
  *src_out = "#include \"bytes_kernel.hpp\"\n" + jit_shape_source(L, offs3, rx, ry, 0) +
             "namespace sth {\ntemplate __global__ void bytes_kernel<" + targs + ">(MapParams);\n}  // namespace sth\n";
  *expr_out = "&sth::bytes_kernel<" + targs + ">";
  return true;
}

inline const JitKernel* jit_bytes_kernel(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int ky,
                                         std::string* why) {
  const JitRequest request = JitRequest('b').add(dtype).add(opk).add(rx).add(ry).add(ky).add(offs3, 3 * static_cast<size_t>(L));
  return jit_remembered(request, [&]() -> const JitKernel* {
    std::string src, expr;
    if (!jit_bytes_source(dtype, opk, L, offs3, rx, ry, ky, &src, &expr)) {
      *why = "no type name";
      return nullptr;
    }
    return jit_load(src, expr, "bytes" + std::to_string(ky), why);
  });
}

// One pass of a multi-array gather as a streaming kernel over one stencil
// argument: its fold f (scaled by its coefficient when `scaled`), combined
// into the running value -- read back from dest (`acc_in`), or started from
// the leading centre terms -- and followed by the centre terms up to the next
// stencil argument, each `coef * A[I]` or `A[I]`, folded left with + or * in
// the element type as the reference's `a + b + c` is.  `items` lists the
// pass's terms in order: 'f' / 'F' the fold (plain / scaled), 'c' / 'C' a
// centre term (plain / scaled), the k-th centre term reading slot k of the
// pass's parameters; the coefficients are parameters too.
struct MultiEpiParams {
  const void* acc;         // dest, read back when the pass continues a fold
  int64_t acc_s1, acc_s2;
  const void* base[8];     // centre arguments (interior element (0,0,0))
  int64_t s1[8], s2[8];
  double coef[8];          // coef[0]: the fold's; coef[1 + k]: centre term k's
};
// The loop of a multi-array epilogue over a lane's V results of one row.
// `rows` are the row pointers (type const T*) of the arrays it reads at the
// result's cells; when the lane's V cells lie inside the row they are read as
// one vector per array, otherwise cell by cell.  `cell(val)` gives the
// statements for one cell (index i, its fold value `f`), `val(k)` the
// expression of array k's value there.
inline std::string jit_epilogue_loop(const std::vector<std::string>& rows,
                                     const std::function<std::string(const std::function<std::string(size_t)>&)>& cell) {
  std::string s;
  for (size_t k = 0; k < rows.size(); ++k)
    s += "    const T* const row" + std::to_string(k) + " = " + rows[k] + ";\n";
  s += "    if (x0 + V <= n0) {\n";
  for (size_t k = 0; k < rows.size(); ++k)
    s += "      const RawVec<T, V> vec" + std::to_string(k) + " = load_vec<T, V>(row" + std::to_string(k) + " + x0);\n";
  s += "#pragma unroll\n"
       "      for (int i = 0; i < V; ++i) {\n"
       "        const T f = out.e[i];\n"
       "        (void)f;\n";
  s += cell([](size_t k) { return "vec" + std::to_string(k) + ".e[i]"; });
  s += "      }\n"
       "    } else {\n"
       "#pragma unroll\n"
       "      for (int i = 0; i < V; ++i) {\n"
       "        if (x0 + i < n0) {\n"
       "          const T f = out.e[i];\n"
       "          (void)f;\n";
  s += cell([](size_t k) { return "row" + std::to_string(k) + "[x0 + i]"; });
  s += "        }\n"
       "      }\n"
       "    }\n";
  return s;
}

// The source and kernel expression of one such pass (false: no type name).
inline bool jit_multi_source(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int rz, int v, int ky,
                             bool acc_in, const std::string& items, bool mul, std::string* src_out,
                             std::string* expr_out) {
  const char* tn = jit_type_name(dtype);
  if (!tn) return false;
  const bool fl = dtype == STH_F32 || dtype == STH_F64;
  auto comb = [&](const std::string& a, const std::string& b) {
    if (fl) return a + (mul ? " * " : " + ") + b;
    return "static_cast<T>(static_cast<U>(static_cast<U>(" + a + ")" + (mul ? " * " : " + ") + "static_cast<U>(" +
           b + ")))";
  };
  std::vector<std::string> rows;  // the running value (passes after the first), then the centre arguments
  if (acc_in) rows.push_back("reinterpret_cast<const T*>(e.acc) + z * e.acc_s2 + y * e.acc_s1");
  for (char c : items)
    if (c == 'c' || c == 'C') {
      const std::string k = std::to_string(rows.size() - (acc_in ? 1 : 0));
      rows.push_back("reinterpret_cast<const T*>(e.base[" + k + "]) + z * e.s2[" + k + "] + y * e.s1[" + k + "]");
    }
  const std::string loop = jit_epilogue_loop(rows, [&](const std::function<std::string(size_t)>& val) {
    std::string b;
    bool first = !acc_in;
    size_t r = 0;
    if (acc_in) b += "        T acc = " + val(r++) + ";\n";
    int k = 0;
    for (char c : items) {
      std::string x;
      if (c == 'f' || c == 'F') {
        x = c == 'F' ? "static_cast<T>(static_cast<T>(e.coef[0]) * f)" : "f";
      } else {
        x = c == 'C' ? "static_cast<T>(static_cast<T>(e.coef[" + std::to_string(k + 1) + "]) * " + val(r) + ")"
                     : val(r);
        ++r;
        ++k;
      }
      if (first) {
        b += "        T acc = " + x + ";\n";
        first = false;
      } else {
        b += "        acc = " + comb("acc", x) + ";\n";
      }
    }
    return b + "        out.e[i] = acc;\n";
  });
  const std::string targs = std::string(tn) + ", " + std::to_string(opk) + ", sth::jit::Shape, " +
                            std::to_string(v) + ", " + std::to_string(ky) + ", sth::jit::Epi";
  const std::string src =
      "#include \"stream_kernel.hpp\"\n" + jit_shape_source(L, offs3, rx, ry, rz) +
      "namespace sth {\nnamespace jit {\n"
      "struct EpiParams {\n"
      "  const void* acc;\n  int64_t acc_s1, acc_s2;\n  const void* base[8];\n  int64_t s1[8], s2[8];\n"
      "  double coef[8];\n};\n"
      "struct Epi {\n"
      "  using Params = EpiParams;\n"
      "  static constexpr bool kStore = true;\n"
      "  Params e;\n"
      "  template <typename R, int V>\n"
      "  __device__ __forceinline__ void apply(RawVec<R, V>& out, int64_t x0, int64_t y, int64_t z, int64_t n0,\n"
      "                                        int) const {\n"
      "    using T = R;\n" + std::string(fl ? "" : "    using U = typename Elem<T>::uacc;\n") + loop +
      "  }\n};\n}  // namespace jit\n"
      "template __global__ void stream_kernel_epi<" + targs + ">(MapParams, jit::EpiParams);\n"
      "}  // namespace sth\n";
  *src_out = src;
  *expr_out = "&sth::stream_kernel_epi<" + targs + ">";
  return true;
}

inline const JitKernel* jit_multi_pass(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int rz, int v,
                                       int ky, bool acc_in, const std::string& items, bool mul, std::string* why) {
  const JitRequest request = JitRequest('m')
                                 .add(dtype).add(opk).add(rx).add(ry).add(rz).add(v).add(ky).add(acc_in).add(mul)
                                 .add(items.data(), items.size())
                                 .add(offs3, 3 * static_cast<size_t>(L));
  return jit_remembered(request, [&]() -> const JitKernel* {
    static_assert(sizeof(MultiEpiParams) == 8 + 16 + 64 + 128 + 64, "epilogue parameter layout");
    std::string src, expr;
    if (!jit_multi_source(dtype, opk, L, offs3, rx, ry, rz, v, ky, acc_in, items, mul, &src, &expr)) {
      *why = "no type name";
      return nullptr;
    }
    return jit_load(src, expr, "multi" + std::to_string(v) + "x" + std::to_string(ky), why);
  });
}

// A stencil argument of a fused multi-array kernel: its fold and shape.
struct JitFold {
  int opk, L, rx, ry, rz;
  const int8_t* offs3;  // L packed (dx, dy, dz)
};

// The source of a multi-array kernel that runs every argument in one pass:
// one stream_body per stencil argument, in call order, each with an
// epilogue that combines its fold and the centre terms up to the next
// stencil argument into registers (`items`, one letter per argument in call
// order: 'f' fold, 'F' scaled fold, 'c' centre value, 'C' scaled centre
// value); the last one's result is stored.  Every value is rounded as in the
// one-pass-per-argument kernels, so the results are the same.
inline bool jit_multi_fused_source(int dtype, int v, int ky, const std::vector<JitFold>& folds,
                                   const std::string& items, bool mul, std::string* src_out, std::string* expr_out) {
  const char* tn = jit_type_name(dtype);
  if (!tn || folds.size() < 2 || folds.size() > STH_MAX_TERMS || items.size() > STH_MAX_TERMS) return false;
  const bool fl = dtype == STH_F32 || dtype == STH_F64;
  auto comb = [&](const std::string& a, const std::string& b) {
    if (fl) return a + (mul ? " * " : " + ") + b;
    return "static_cast<T>(static_cast<U>(static_cast<U>(" + a + ")" + (mul ? " * " : " + ") + "static_cast<U>(" +
           b + ")))";
  };
  std::vector<size_t> at;  // position of each fold in `items`
  for (size_t u = 0; u < items.size(); ++u)
    if (items[u] == 'f' || items[u] == 'F') at.push_back(u);
  if (at.size() != folds.size()) return false;
  std::string src = "#include \"stream_kernel.hpp\"\n";
  for (size_t f = 0; f < folds.size(); ++f)
    src += jit_shape_source(folds[f].L, folds[f].offs3, folds[f].rx, folds[f].ry, folds[f].rz,
                            "Shape" + std::to_string(f));
  src += "namespace sth {\nnamespace jit {\nusing T = " + std::string(tn) + ";\nconstexpr int kV = " +
         std::to_string(v) + ", kKY = " + std::to_string(ky) + ";\n";
  std::string calls;
  int nc = 0;
  for (size_t f = 0; f < folds.size(); ++f) {
    const bool last = f + 1 == folds.size();
    const size_t lo = f == 0 ? 0 : at[f], hi = last ? items.size() : at[f + 1];
    std::vector<std::string> rows;  // the centre arguments of items lo .. hi - 1
    for (size_t u = lo; u < hi; ++u)
      if (items[u] == 'c' || items[u] == 'C') {
        const std::string k = std::to_string(nc++);
        rows.push_back("reinterpret_cast<const T*>(P.cbase[" + k + "]) + z * P.cs2[" + k + "] + y * P.cs1[" + k + "]");
      }
    const std::string loop = jit_epilogue_loop(rows, [&](const std::function<std::string(size_t)>& val) {
      std::string b;
      bool first = f == 0;
      if (!first) b += "        T a = acc[j][i];\n";
      size_t r = 0;
      for (size_t u = lo; u < hi; ++u) {
        const char c = items[u];
        const std::string cu = "static_cast<T>(P.coef[" + std::to_string(u) + "])";
        std::string x;
        if (c == 'f' || c == 'F') {
          x = c == 'F' ? "static_cast<T>(" + cu + " * f)" : "f";
        } else {
          x = c == 'C' ? "static_cast<T>(" + cu + " * " + val(r) + ")" : val(r);
          ++r;
        }
        if (first) {
          b += "        T a = " + x + ";\n";
          first = false;
        } else {
          b += "        a = " + comb("a", x) + ";\n";
        }
      }
      return b + (last ? "        out.e[i] = a;\n" : "        acc[j][i] = a;\n");
    });
    const std::string e = "E" + std::to_string(f);
    src += "struct " + e + " {\n"
           "  static constexpr bool kStore = " + std::string(last ? "true" : "false") + ";\n"
           "  const StreamMultiParams& P;\n"
           "  T (&acc)[kKY][kV];\n"
           "  template <typename R, int V>\n"
           "  __device__ __forceinline__ void apply(RawVec<R, V>& out, int64_t x0, int64_t y, int64_t z, int64_t n0,\n"
           "                                        int j) const {\n" +
           std::string(fl ? "" : "    using U = typename Elem<T>::uacc;\n") + loop + "  }\n};\n";
    calls += "  stream_body<T, " + std::to_string(folds[f].opk) + ", Shape" + std::to_string(f) +
             ", kV, kKY>(P.term[" + std::to_string(f) + "], bx, by, bz, lane, wave, " + e + "{P, acc});\n";
  }
  src += "__global__ __launch_bounds__(256) void multi_stream_kernel(StreamMultiParams P) {\n"
         "  const int nblocks = P.tiles_x * P.tiles_y * P.tiles_z;\n"
         "  const int bid = xcd_block_id(static_cast<int>(blockIdx.x), nblocks, P.xcd_remap);\n"
         "  const int bx = bid % P.tiles_x;\n"
         "  const int byz = bid / P.tiles_x;\n"
         "  const int by = byz % P.tiles_y;\n"
         "  const int bz = byz / P.tiles_y;\n"
         "  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);\n"
         "  const int lane = static_cast<int>(threadIdx.x) & 63;\n"
         "  T acc[kKY][kV];\n" +
         calls + "}\n}  // namespace jit\n}  // namespace sth\n";
  *src_out = src;
  *expr_out = "&sth::jit::multi_stream_kernel";
  return true;
}

inline const JitKernel* jit_multi_fused(int dtype, int v, int ky, const std::vector<JitFold>& folds,
                                        const std::string& items, bool mul, std::string* why) {
  std::string src, expr;
  if (!jit_multi_fused_source(dtype, v, ky, folds, items, mul, &src, &expr)) {
    *why = "no type name or too many terms";
    return nullptr;
  }
  return jit_load(src, expr, "mfused" + std::to_string(v) + "x" + std::to_string(ky), why);
}

// Launch a multi-array pass: the call's parameters and the epilogue's.
inline hipError_t jit_launch_multi(hipFunction_t fn, const MapParams& p, const MultiEpiParams& e, hipStream_t s) {
  const unsigned nblocks = static_cast<unsigned>(p.tiles_x) * p.tiles_y * p.tiles_z;
  void* args[] = {const_cast<MapParams*>(&p), const_cast<MultiEpiParams*>(&e)};
  return hipModuleLaunchKernel(fn, nblocks, 1, 1, 256, 1, 1, 0, s, args, nullptr);
}

// Rows per wave of the 3-D two-step kernel for storage type `dtype` (its
// staged value's size decides, as zmarch2_rows does on the device).
inline int jit_zmarch2_rows(int dtype) {
  const bool wide = dtype == STH_F64 || dtype == STH_I64 || dtype == STH_U64;  // 8-byte staged values
  return wide ? 10 : 16;
}

// Most steps per launch of the 2-D multi-step kernel for storage type
// `dtype`, as ymarch_gens gives it on the device.
inline int jit_ymarch_gens(int dtype, int L) {
  const bool half = dtype == STH_BF16 || dtype == STH_F16 || dtype == STH_I16 || dtype == STH_U16;
  return half ? 4 : (L <= 4 ? 8 : 6);
}

// The source of a multi-step kernel (temporal blocking) specialised to one
// radius-1 shape: ymarch_kernel (2-D) or zmarch2_kernel (3-D) for
// boundary `bc` (false: no type name).
inline bool jit_fused_source(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int rz, int ndim, int bc,
                             int gens, std::string* src_out, std::string* expr_out) {
  const char* tn = jit_type_name(dtype);
  if (!tn) return false;
  const std::string head = std::string(tn) + ", " + std::to_string(opk) + ", sth::jit::Shape, ";
  const std::string targs = ndim == 3 ? head + std::to_string(jit_zmarch2_rows(dtype)) + ", " + std::to_string(bc)
                                      : head + std::to_string(gens) + ", " + std::to_string(bc);
  const std::string kern = ndim == 3 ? "zmarch2_kernel" : "ymarch_kernel";
  *src_out = "#include \"ymarch_kernel.hpp\"\n" + jit_shape_source(L, offs3, rx, ry, rz) +
             "namespace sth {\ntemplate __global__ void " + kern + "<" + targs + ">(MapParams);\n}  // namespace sth\n";
  *expr_out = "&sth::" + kern + "<" + targs + ">";
  return true;
}

inline const JitKernel* jit_fused_kernel(int dtype, int opk, int L, const int8_t* offs3, int rx, int ry, int rz,
                                         int ndim, int bc, int gens, std::string* why) {
  const JitRequest request = JitRequest('f').add(dtype).add(opk).add(rx).add(ry).add(rz)
                                 .add(ndim).add(bc).add(gens).add(offs3, 3 * static_cast<size_t>(L));
  return jit_remembered(request, [&]() -> const JitKernel* {
    std::string src, expr;
    if (!jit_fused_source(dtype, opk, L, offs3, rx, ry, rz, ndim, bc, gens, &src, &expr)) {
      *why = "no type name";
      return nullptr;
    }
    return jit_load(src, expr, ndim == 3 ? "zmarch2" : "ymarch", why);
  });
}

// The scatter kernel with the interior order of each dest-column residue as
// code: `deltas` holds, per residue r = 0..S-1, the L LDS deltas of the
// senders in arrival order (the table the build-time kernel reads from LDS).
inline bool jit_scatter_source(int dtype, int kind, int combine, int S, int L, const int32_t* deltas,
                               std::string* src_out, std::string* expr_out) {
  const char* tn = jit_type_name(dtype);
  if (!tn || (dtype != STH_F32 && dtype != STH_F64)) return false;
  std::string cases;
  for (int r = 0; r < S; ++r) {
    cases += "      case " + std::to_string(r) + ":\n";
    for (int t = 0; t < L; ++t)
      cases += "        acc = scatter_step<T, KIND, COMB, " + std::to_string(deltas[r * L + t]) +
               ">(acc, cf, la, lb, c, bd);\n";
    cases += "        break;\n";
  }
  const std::string targs = std::string(tn) + ", " + std::to_string(kind) + ", " + std::to_string(combine) +
                            ", sth::jit::ScatterOrder";
  *src_out =
      "#include \"scatter_kernel.hpp\"\n"
      "namespace sth {\nnamespace jit {\n"
      "struct ScatterOrder {\n"
      "  static constexpr bool kStatic = true;\n"
      "  template <typename T, int KIND, int COMB>\n"
      "  __device__ __forceinline__ static T run(int r, T acc, T cf, const T* __restrict__ la,\n"
      "                                          const T* __restrict__ lb, int c) {\n"
      "    T bd = T(0);\n"
      "    if constexpr (KIND >= STH_SCATTER_DOWNHILL) bd = lb[c];\n"
      "    switch (r) {\n" + cases + "      default: break;\n    }\n    return acc;\n  }\n};\n"
      "}  // namespace jit\n"
      "template __global__ void scatter_kernel<" + targs + ">(ScatterParams, const int32_t*);\n"
      "}  // namespace sth\n";
  *expr_out = "&sth::scatter_kernel<" + targs + ">";
  return true;
}

inline const JitKernel* jit_scatter_kernel(int dtype, int kind, int combine, int S, int L, const int32_t* deltas,
                                           std::string* why) {
  const JitRequest request = JitRequest('c').add(dtype).add(kind).add(combine).add(S).add(deltas, static_cast<size_t>(S) * L);
  return jit_remembered(request, [&]() -> const JitKernel* {
    std::string src, expr;
    if (!jit_scatter_source(dtype, kind, combine, S, L, deltas, &src, &expr)) {
      *why = "no specialisation for this element type";
      return nullptr;
    }
    return jit_load(src, expr, "scatter", why);
  });
}

// Launch a loaded specialisation with the call's parameters (one block of
// 256 threads per tile, as launch_stream does).
inline hipError_t jit_launch(hipFunction_t fn, const MapParams& p, hipStream_t s) {
  const unsigned nblocks = static_cast<unsigned>(p.tiles_x) * p.tiles_y * p.tiles_z;
  void* args[] = {const_cast<MapParams*>(&p)};
  return hipModuleLaunchKernel(fn, nblocks, 1, 1, 256, 1, 1, 0, s, args, nullptr);
}

}  // namespace sth
