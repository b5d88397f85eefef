// run_routes.cpp — sage_run and sage_flash_run on a host without a GPU: the C
// ABI of sage_attn_fwd.hip with stand-ins that write down the pre-pass call
// and the kernel launch they are asked for, one JSON object each, and do
// nothing else.  Linked with libsage_attn.so for the size queries.
#include <string>

#include "../../tribench_amd/csrc/sage_attn_fwd.hip"

static thread_local std::string routes;

static void field(const char* name, long long x) { routes += std::string(", \"") + name + "\": " + std::to_string(x); }
static void field3(const char* name, const int64_t* s) {
  routes += std::string(", \"") + name + "\": " +
            (s ? "[" + std::to_string(s[0]) + ", " + std::to_string(s[1]) + ", " + std::to_string(s[2]) + "]" : "null");
}
static int launch(const char* kernel, const sage::AttnArgs& a, int nw) {
  routes += std::string("{\"launch\": \"") + kernel + "\"";
  field("nw", nw);
  field("wpe", nw == 4 && a.wpe == 3 ? 3 : 2);
  field("grp", a.grp ? a.grp : 1);
  field("nsplit", a.nsplit ? a.nsplit : 1);
  field("vrow", a.vrow);
  const int64_t sq[3] = {a.sq[0], a.sq[1], a.sqn};
  field3("q_strides", sq);
  field("q8_out", (long long)a.q8_out);
  routes += "}\n";
  return 0;
}

namespace sage {
int launch_attn_i8(const AttnArgs& a, int, int, int, int nw, hipStream_t, const char*) { return launch("i8", a, nw); }
int launch_attn_i8q(const AttnArgs& a, int, int, int, int nw, hipStream_t, const char*) { return launch("i8q", a, nw); }
int launch_attn_flash(const AttnArgs& a, int, int, int nw, hipStream_t, const char*) { return launch("flash", a, nw); }
int launch_attn_part(const AttnArgs& a, int, int, bool i8, int, hipStream_t, const char*) {
  return launch(i8 ? "i8 part" : "flash part", a, 4);
}
int prepass_any(const char*, const void* q, const void*, const void* v, int, int64_t, int64_t, int64_t, int64_t,
                int64_t, int64_t, const int64_t*, const int64_t*, const int64_t*, float, int, int, int, int, int,
                int8_t* q8, const int64_t* q8_strides, float*, int8_t* k8, const int64_t* k8_strides, float*, float*,
                uint8_t*, const int64_t*, float*, void*, size_t, int, void*, size_t, void*) {
  routes += "{\"launch\": \"prepass\"";
  field("quant_q", q != nullptr);
  field("v", v != nullptr);
  field("q8", (long long)q8);
  field3("q8_strides", q8_strides);
  field("k8", (long long)k8);
  field3("k8_strides", k8_strides);
  routes += "}\n";
  return 0;
}
}  // namespace sage

// what the calls since the last one of this function did
extern "C" const char* take_routes() {
  static thread_local std::string out;
  out.swap(routes);
  routes.clear();
  return out.c_str();
}

extern "C" int k_waves_pay(int64_t nblk, int64_t D, int vt_in_b, int pv_mode) {
  return sage::k_waves_pay(nblk, D, vt_in_b, pv_mode);
}
