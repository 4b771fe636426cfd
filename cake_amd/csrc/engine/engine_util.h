// Host helpers shared by the native engines (llama_engine.cpp, sd_engine.cpp): HIP error
// checks, the package directory, file reads and the GEMM tile planner (ops/gemm.py plan()).
#pragma once

#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <fstream>
#include <sstream>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../runtime/json.h"
#include "../runtime/net.h"

namespace cake {

struct Error : std::runtime_error {
  using std::runtime_error::runtime_error;
};

inline void hip_check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw Error(std::string(what) + ": " + hipGetErrorString(e));
}
inline void k_check(int rc, const char* what) {
  if (rc == 0) return;
  if (rc >= 1000)  // driver/blaslt.cpp: 1000 + hipblasStatus_t
    throw Error(std::string(what) + ": hipBLASLt status " + std::to_string(rc - 1000));
  throw Error(std::string(what) + ": " + hipGetErrorString((hipError_t)rc));
}

// ---------------------------------------------------------------------------
// control plane of the multi-rank engines: IPC handles as hex, JSON frames over TCP
// ---------------------------------------------------------------------------
inline std::string hex_of(const void* p, size_t n) {
  static const char* d = "0123456789abcdef";
  std::string s;
  const uint8_t* b = static_cast<const uint8_t*>(p);
  for (size_t i = 0; i < n; ++i) {
    s.push_back(d[b[i] >> 4]);
    s.push_back(d[b[i] & 15]);
  }
  return s;
}

inline void unhex(const std::string& s, void* out, size_t n) {
  if (s.size() != 2 * n) throw Error("bad IPC handle");
  auto v = [](char c) { return c <= '9' ? c - '0' : c - 'a' + 10; };
  uint8_t* b = static_cast<uint8_t*>(out);
  for (size_t i = 0; i < n; ++i) b[i] = (uint8_t)(v(s[2 * i]) << 4 | v(s[2 * i + 1]));
}

inline void send_json(int fd, const Json& j) {
  const std::string t = j.dump();
  send_frame(fd, reinterpret_cast<const uint8_t*>(t.data()), (uint32_t)t.size());
}
inline Json recv_json(int fd) { return Json::parse(recv_frame(fd)); }

// <root>/cake_amd/lib/libcake_engine.so -> <root>/cake_amd
inline std::string pkg_dir() {
  Dl_info info{};
  if (dladdr(reinterpret_cast<void*>(&pkg_dir), &info) && info.dli_fname) {
    char buf[4096];
    const char* p = realpath(info.dli_fname, buf);
    std::string s = p ? p : info.dli_fname;
    for (int i = 0; i < 2; ++i) {
      const auto cut = s.find_last_of('/');
      if (cut == std::string::npos) return ".";
      s = s.substr(0, cut);
    }
    return s;
  }
  return ".";
}

inline std::string read_file(const std::string& path) {
  std::ifstream f(path, std::ios::binary);
  if (!f) throw Error("cannot read " + path);
  std::stringstream ss;
  ss << f.rdbuf();
  return ss.str();
}

// ---------------------------------------------------------------------------
// GEMM tile plan (ops/gemm.py resolve(): measured table, else the kernel library's estimate)
// ---------------------------------------------------------------------------
// plan cfg naming the library GEMM (hipBLASLt, driver/blaslt.cpp; ops/gemm.py LIB).
// Off the default path: table entries naming it are read only under CAKE_GEMM_LIB=1
// (the A/B arm of scripts/bench_gemm_lib.py); otherwise every shape runs an MFMA plan.
constexpr int kGemmLib = -1;
inline bool gemm_lib_enabled() {
  const char* e = std::getenv("CAKE_GEMM_LIB");
  return e && *e == '1';
}

extern "C" int cake_gemm_plan(int M, long long Nv, int K, int epi, int big, int* cfg, int* splits);

struct GemmPlanner {
  struct Tuned { long long M, Nv, K; std::string epi; int cfg, splits; };
  std::vector<Tuned> tuned;

  void load(std::string path) {  // CAKE_GEMM_TABLE overrides (A/B of plan tables)
    if (const char* e = std::getenv("CAKE_GEMM_TABLE"); e && *e) path = e;
    std::ifstream f(path);
    if (!f) return;
    const bool lib_ok = gemm_lib_enabled();
    try {
      const Json j = Json::parse(read_file(path));
      static const int known[] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27,
                                  28, 29, 30, 31, 32, 33, 34, 35, 36, 37, 38};
      for (const auto& e : j.get("entries").items()) {
        const int cfg = (int)e.get("cfg").as_int();
        const std::string ep = e.get("epi").as_string();
        const bool lib = lib_ok && cfg == kGemmLib && (ep == "store" || ep == "resid32" || ep == "store32" ||
                                             ep == "swiglu");
        if (!lib && std::find(std::begin(known), std::end(known), cfg) == std::end(known)) continue;
        tuned.push_back({e.get("M").as_int(), e.get("Nv").as_int(), e.get("K").as_int(),
                         e.get("epi").as_string(), cfg, (int)e.get("splits").as_int()});
      }
    } catch (const std::exception&) {
      tuned.clear();  // a malformed table only loses the measured overrides
    }
  }

  bool has_lib() const {
    for (const auto& e : tuned)
      if (e.cfg == kGemmLib) return true;
    return false;
  }

  // the plan that runs (ops/gemm.py resolve): the measured entry of this very size unless the
  // kernel library's estimate puts it well behind, else the estimate's best; epi_id: its epilogue id;
  // mfma_only: as if no plan named the library GEMM
  std::pair<int, int> resolve(long long M, long long Nv, long long K, const std::string& epi, int epi_id,
                              bool big, bool mfma_only = false) const {
    int cfg = -1, splits = 1;
    for (const auto& e : tuned)
      if (e.M == M && e.Nv == Nv && e.K == K && e.epi == epi && !(mfma_only && e.cfg == kGemmLib)) {
        if (e.cfg == kGemmLib) return {kGemmLib, 1};
        cfg = e.cfg;
        splits = e.splits;
        break;
      }
    cake_gemm_plan((int)M, Nv, (int)K, epi_id, big ? 1 : 0, &cfg, &splits);
    return {cfg, splits};
  }
};

}  // namespace cake
