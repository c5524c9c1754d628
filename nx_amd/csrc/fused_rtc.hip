// Fused element-wise groups compiled at run time, one kernel per distinct program.
//
// The interpreting kernels of fused.hip decode each instruction for every vector of eight elements:
// scalar work that costs more than the arithmetic of a short chain.  Here the same program is
// written out as compile-time constants over the same device functions (fused_ops.cuh) and given
// to the run-time compiler once; the kernel is kept per context, keyed by what it is specialised on.  Same
// functions, same order, same flags (no contraction, no packed f32): bit-identical results.
// The device headers are embedded in the library as text, so nothing is read from disk.
#include <hip/hiprtc.h>

#include <algorithm>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "fused_ops.cuh"
#include "internal.h"
#include "rtc_headers.inc"

namespace hipnx {

// what the device headers take from host headers when the offline compiler builds them
static const char *const RTC_PREAMBLE = R"(
typedef unsigned char uint8_t; typedef signed char int8_t; typedef unsigned short uint16_t; typedef short int16_t;
typedef unsigned int uint32_t; typedef int int32_t; typedef unsigned long uint64_t; typedef long int64_t;
typedef unsigned long uintptr_t;
#define NAN __builtin_nanf("")
#define INFINITY __builtin_inff()
#define INT64_MAX 9223372036854775807L
#define INT64_MIN (-INT64_MAX - 1)
namespace std {
template <bool B, class T, class F> struct conditional { typedef T type; };
template <class T, class F> struct conditional<false, T, F> { typedef F type; };
template <class A, class B> struct is_same { static constexpr bool value = false; };
template <class A> struct is_same<A, A> { static constexpr bool value = true; };
template <class T> struct is_floating_point { static constexpr bool value = false; };
template <> struct is_floating_point<float> { static constexpr bool value = true; };
template <> struct is_floating_point<double> { static constexpr bool value = true; };
}
#include "fused_ops.cuh"
)";

static void list_of(std::string &s, const char *name, const char *type, int n, const std::function<std::string(int)> &at) {
  s += std::string("  static constexpr ") + type + " " + name + "[] = {";
  for (int i = 0; i < (n > 0 ? n : 1); i++) s += (i ? ", " : "") + (n > 0 ? at(i) : std::string("0"));
  s += "};\n";
}

// What the lanes of a stage program keep in registers between stages: element values carried from one stage to the next,
// and an input that several stages read.
struct Keeps {
  int form = ROW_WHOLE, tail = 0;  // how lanes share a row (fused_ops.cuh), elements behind the vectors of a ROW_LANE row
  int tpr = 0;          // lanes per row, 0 where the kernel does not take rows one by one
  int trips = 0;        // vectors of a lane along a row, 0 when nothing is kept
  bool carries = false;
  bool written_out = false;  // a lane's trips as straight code (fused_ops.cuh, for_each_vector)
  int held = -1;        // the input, and the first stage that reads it
  int held_stage = -1;
};
// What a function costs a trip that is written out: the branches it has per element and its code for a vector of eight in KB,
// read off the compiler's output (the others: no branch, 1 KB or less).
struct Cost {
  int branches, kbytes;
};
static Cost cost_of(const hipnx_fused_instr &q) {
  if (q.kind == HIPNX_FUSED_UNARY) switch (q.op) {
    case HIPNX_TANH: return {1, 2};
    case HIPNX_ERF: return {1, 3};
    case HIPNX_SIN: case HIPNX_COS: case HIPNX_TAN: return {2, 7};
    case HIPNX_ERF_INV: return {4, 9};
    case HIPNX_SIGMOID: case HIPNX_EXPM1: case HIPNX_RSQRT: return {0, 2};
    case HIPNX_ERFC: return {0, 3};
    case HIPNX_SINH: case HIPNX_COSH: return {0, 4};
    case HIPNX_LOG1P: case HIPNX_ASINH: case HIPNX_ACOSH: case HIPNX_ATANH: return {0, 5};
  }
  if (q.kind == HIPNX_FUSED_BINARY) switch (q.op) {
    case HIPNX_REMAINDER: return {3, 2};
    case HIPNX_ATAN2: return {0, 3};
    case HIPNX_POW: return {0, 7};
  }
  return {0, 0};
}

// Lanes per row and their shares: those of the separate reduction of rows of that length, whose order the stages keep (run_reduce_t
// of reduce_kernels.cuh).  `walk`: the kernel takes the rows one by one (stages, or rows that are not whole vectors).
static int class_lanes(const FusedArgs &a) { return a.cols > 4096 ? FBLOCK : WAVE; }
static void share_row(const FusedArgs &a, bool walk, Keeps &k) {
  if (!walk) return;
  k.tpr = class_lanes(a);
  // (a wave per row of 64 had an eighth of its lanes at work)
  if (a.cols <= 256) k.tpr = a.cols <= 16 ? 1 : a.cols <= 64 ? 8 : a.cols <= 128 ? 16 : 32;
  // (a contraction's rows are in LDS: with up to four vectors a lane, two or four rows share a wave's reductions, which are a fifth of
  // the instructions when a row of 512 takes it alone; the order of a sum is this kernel's own.
  // bf16 4 x 8 x 512 x 512: 20.9 -> 19.3 us a pass.  One row alone -- a step of decoding -- is faster with a wave: 784 columns 7.7, 9.9 so)
  if (a.scores >= 0 && a.cols > 256 && a.scores_rows >= 8) k.tpr = a.cols <= 512 ? 16 : a.cols <= 1024 ? 32 : WAVE;
  k.form = a.cols <= 16 ? ROW_LANE : a.cols % FE == 0 ? ROW_WHOLE : a.cols <= 256 ? ROW_GROUP : ROW_RAGGED;
  if (k.form == ROW_LANE) k.trips = (int)(a.cols / FE), k.tail = (int)(a.cols % FE);
}

static Keeps what_is_kept(const FusedArgs &a, bool walk) {
  Keeps k;
  bool stages = false;
  for (int i = 0; i < a.n_instr; i++) stages |= a.ins[i].kind == HIPNX_FUSED_ROW_REDUCE;
  share_row(a, walk, k);
  if (!stages) return k;
  // (one trip more where the elements around the vectors are code of their own)
  const int64_t trips = (a.cols / FE + k.tpr - 1) / k.tpr, written = trips + (a.cols % FE != 0);
  if (trips > 16) return k;  // (the host refuses longer rows for programs that carry values)
  // which stages read an input along the row, and up to which stage a carried value is waiting to be read
  unsigned reads[HIPNX_FUSED_MAX_INPUTS] = {};
  int stage = 0, carried_from = -1;
  bool on_stat = false, rounds = false, rounds_f16 = false;
  Cost trip = {0, 0};
  for (int i = 0; i < a.n_instr; i++) {
    const hipnx_fused_instr &q = a.ins[i];
    if (!on_stat) {
      const Cost c = cost_of(q);
      trip.branches += c.branches, trip.kbytes += c.kbytes;
      rounds_f16 |= q.dt == HIPNX_F16;
      rounds |= q.dt == HIPNX_F16 || q.dt == HIPNX_BF16;
    }
    on_stat = q.kind == HIPNX_FUSED_ROW_REDUCE || (on_stat && q.kind != HIPNX_FUSED_ROW_STAT);
    // (a SET or BINARY on integers reads the words as they are in memory; a SELECT reads floats whatever its flags:
    // the cases of fetch_static)
    const bool raw = (q.flags & HIPNX_FUSED_FLAG_INT) != 0 && q.kind != HIPNX_FUSED_SELECT;
    auto source = [&](int src, int arg) {
      if (src == HIPNX_FUSED_SRC_CARRY) carried_from = stage - 1;  // (the last stage that leaves a value somebody reads)
      if (src == HIPNX_FUSED_SRC_INPUT && a.in_cs[arg] == 1 && !raw) reads[arg] |= 1u << stage;
    };
    if (q.kind == HIPNX_FUSED_SET || q.kind == HIPNX_FUSED_BINARY || q.kind == HIPNX_FUSED_SELECT) source(q.src, q.arg);
    if (q.kind == HIPNX_FUSED_SELECT) source(q.src2, q.arg2);
    if (q.kind == HIPNX_FUSED_ROW_STAT) stage++;
  }
  k.carries = carried_from >= 0;
  if (k.carries) k.trips = (int)trips;
  // Written-out trips gain where the compiler can lay one trip's loads and arithmetic over the next's, and hold the row for
  // one read (a layer norm of sigmoids, f32 4096 x 4096: 57 us as a loop, 38 written out).  A branch per element ends
  // that, and the straight code then costs its own fetching.  f32, loop / written out: tanh in two stages, 3 trips 36 / 30 us,
  // 4 trips 34 / 33, 6 trips 35 / 40, 8 trips 39 / 56; erf 3 trips 39 / 40, 4 trips 39 / 44, 8 trips 44 / 79; sin 8 trips 38 / 104.
  // With 16-bit roundings there is less to gain: tanh in one stage, bf16, 2 trips 26 / 28, 4 trips 26 / 29; and in f16, whose
  // conversions are instructions too, nothing once a function is long (atan2, 2 to 16 trips, 1 to 8 % slower).
  // And the code has to stay near what the instruction cache holds (64 KB for two CUs): pow in two stages, 16 trips (240 KB),
  // 154 / 172 us, and 2.4 s to compile instead of 0.5.
  if (trip.branches * written > (rounds ? 1 : 6) || trip.kbytes * written > 96 || (rounds_f16 && trip.kbytes > 0)) return k;
  // Carried values alone gain only where the compiler leaves the loop over them rolled: f32, logarithms, 14 trips 37 / 43 us,
  // 16 trips 51 / 46; square roots, 15 trips 32 / 35, 16 trips 40 / 37.
  k.written_out = k.carries && trips > 15;
  for (int in = 0; in < a.n_inputs; in++) {
    if (!(reads[in] & (reads[in] - 1)) || k.held >= 0) continue;  // one stage reads it: nothing to gain
    // a lane has room for 16 vectors (128 of its registers): an input that is still read once a carried value is there
    // shares them
    const int last = 31 - __builtin_clz(reads[in]);
    if (carried_from >= 0 && last > carried_from && trips > 8) continue;
    k.trips = (int)trips;
    k.written_out = true;
    k.held = in;
    k.held_stage = __builtin_ctz(reads[in]);
  }
  return k;
}

// everything a compiled kernel is specialised on, as bytes: the cache key.  What the length of a row decides comes last: the keys of
// one program's kernels for rows of other lengths differ in it alone.
constexpr size_t LENGTH_KEY = 4 * sizeof(int);
// columns of a contraction's result that LDS has room for: whole steps of 512, one kernel for all lengths of a step
static int scores_class(const FusedArgs &a) { return a.scores < 0 ? 0 : (int)((a.cols + 511) / 512 * 512); }
static std::string make_key(const FusedArgs &a, const Keeps &keeps, int reduce_op, bool block_per_row, int scores_k) {
  std::string k;
  k.reserve(40 + 16 * a.n_instr + 8 * a.n_inputs);
  const int head[8] = {a.n_instr, a.n_inputs, a.out_dt, reduce_op * 2 + (block_per_row ? 1 : 0), a.words, a.scores, scores_class(a), scores_k};
  k.append((const char *)head, sizeof(head));
  k.append((const char *)a.ins, sizeof(hipnx_fused_instr) * a.n_instr);
  k.append((const char *)a.in_dt, sizeof(int) * a.n_inputs);
  k.append((const char *)a.in_cs, sizeof(int) * a.n_inputs);
  const int length[4] = {keeps.form, keeps.tpr, keeps.tail, keeps.trips};
  static_assert(sizeof(length) == LENGTH_KEY, "the part of the key that a row's length decides");
  k.append((const char *)length, sizeof(length));
  return k;
}

// A program that keeps an input in registers only to read it once could do without, and then takes rows of any number of whole
// vectors (a wave per row, a block per long row): its module also has that kernel, for a capture that meets a length which has
// not been compiled (a new module is no work to record).  One that carries values cannot.
static bool is_for_any_length(const FusedArgs &a, const Keeps &k) { return a.scores < 0 && k.form == ROW_WHOLE && k.trips == 0 && (k.tpr == 0 || k.tpr == class_lanes(a)); }
static bool has_kernel_for_any_length(const FusedArgs &a, const Keeps &k) { return a.scores < 0 && a.cols % FE == 0 && !k.carries && !is_for_any_length(a, k); }
static std::string any_length(const std::string &name) { return name + "_any"; }

// the whole translation unit for one program
static std::string make_source(const FusedArgs &a, const Keeps &keeps, int reduce_op, bool block_per_row, int scores_k, const std::string &name) {
  std::string s = RTC_PREAMBLE;
  s += "namespace hipnx {\nstruct Program {\n  static constexpr int n_instr = " + std::to_string(a.n_instr) + ", out_dt = " + std::to_string(a.out_dt) + ", words = " + std::to_string(a.words) +
       ", scores = " + std::to_string(a.scores < 0 ? -2 : a.scores) + ", scores_cols = " + std::to_string(scores_class(a)) + ", scores_k = " + std::to_string(scores_k) + ";\n";
  const hipnx_fused_instr *q = a.ins;
  list_of(s, "kind", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].kind); });
  list_of(s, "op", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].op); });
  list_of(s, "src", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].src); });
  list_of(s, "arg", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].arg); });
  list_of(s, "src2", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].src2); });
  list_of(s, "arg2", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].arg2); });
  list_of(s, "flags", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].flags); });
  list_of(s, "dt", "int", a.n_instr, [&](int i) { return std::to_string((int)q[i].dt); });
  list_of(s, "imm", "unsigned", a.n_instr, [&](int i) { return std::to_string(q[i].imm_bits) + "u"; });
  list_of(s, "imm2", "unsigned", a.n_instr, [&](int i) { return std::to_string(q[i].imm2_bits) + "u"; });
  list_of(s, "in_dt", "int", a.n_inputs, [&](int k) { return std::to_string(a.in_dt[k]); });
  list_of(s, "in_cs", "int", a.n_inputs, [&](int k) { return std::to_string(a.in_cs[k]); });
  // stages: where each one's reduction and the end of its work on the statistic are (-1, n_instr for the last)
  std::vector<int> seg_red, seg_save;
  for (int i = 0; i < a.n_instr; i++) {
    if (q[i].kind == HIPNX_FUSED_ROW_REDUCE) seg_red.push_back(i);
    if (q[i].kind == HIPNX_FUSED_ROW_STAT) seg_save.push_back(i);
  }
  const bool stages = !seg_red.empty();
  if (seg_save.size() < seg_red.size() || seg_save.empty() || seg_save.back() != a.n_instr - 1) {  // a last, element-wise stage
    seg_red.push_back(-1);
    seg_save.push_back(a.n_instr);
  }
  list_of(s, "seg_red", "int", (int)seg_red.size(), [&](int k) { return std::to_string(seg_red[k]); });
  list_of(s, "seg_save", "int", (int)seg_save.size(), [&](int k) { return std::to_string(seg_save[k]); });
  auto keeping = [&](const char *p, const Keeps &k) {
    return std::string("struct ") + p + " : Program {\n  static constexpr int form = " + std::to_string(k.form) + ", tpr = " + std::to_string(k.tpr) + ", tail = " + std::to_string(k.tail) +
           ";\n  static constexpr bool unal = " + (k.form == ROW_WHOLE && a.words < 0 ? "false" : "true") + ";\n  static constexpr int nv = " + std::to_string(k.trips) + ", written_out = " + std::to_string(k.written_out) + ", held = " + std::to_string(k.held) +
           ", held_stage = " + std::to_string(k.held_stage) + ";\n};\n";
  };
  auto kernel = [&](const std::string &called) {
    return "extern \"C\" __global__ void __launch_bounds__(FBLOCK) " + called + (a.words >= 0 ? "(FusedWordsArgs" : "(FusedArgs") + " by_value) {\n  (void)by_value;\n";
  };
  s += "};\n" + keeping("P", keeps);
  Keeps any;
  any.tpr = class_lanes(a);
  if (has_kernel_for_any_length(a, keeps)) s += keeping("Any", any);
  s += "}\nusing namespace hipnx;\n";
  if (has_kernel_for_any_length(a, keeps)) s += kernel(any_length(name)) + "  fused_row_stages_body<Any>();\n}\n";
  s += kernel(name);
  const char *tpr = block_per_row ? "FBLOCK" : "WAVE";
  if (a.words >= 0) s += "  fused_words_body<P>();\n";
  else if (a.scores >= 0) s += "  fused_scores_body<P>();\n";
  else if (stages || keeps.form != ROW_WHOLE) s += "  fused_row_stages_body<P>();\n";
  else switch (reduce_op) {
    case HIPNX_RED_SUM: s += std::string("  fused_reduce_rows_body<RunStatic<P>, PlainReducer<double, HIPNX_RED_SUM, false>, double, ") + tpr + ">();\n"; break;
    case HIPNX_RED_MAX: s += std::string("  fused_reduce_rows_body<RunStatic<P>, PlainReducer<float, HIPNX_RED_MAX, false>, float, ") + tpr + ">();\n"; break;
    case HIPNX_RED_MIN: s += std::string("  fused_reduce_rows_body<RunStatic<P>, PlainReducer<float, HIPNX_RED_MIN, false>, float, ") + tpr + ">();\n"; break;
    default: s += "  fused_elementwise_body<RunStatic<P>>();\n"; break;
  }
  s += "}\n";
  return s;
}

static int compile(hipnx_ctx *ctx, const std::string &src, const std::string &name, bool with_any, hipnx_ctx::FusedKernel *out) {
  hipDeviceProp_t prop;
  HIPNX_HIP(hipGetDeviceProperties(&prop, ctx->device));
  const std::string arch = std::string("--offload-arch=") + prop.gcnArchName;
  hiprtcProgram prog;
  if (hiprtcCreateProgram(&prog, src.c_str(), "fused_group.hip", RTC_NHEADERS, RTC_HEADER_SOURCES, RTC_HEADER_NAMES) != HIPRTC_SUCCESS)
    return set_error(HIPNX_EHIP, "fused: the run-time compiler did not take the program");
  const char *opts[] = {arch.c_str(), "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
  const hiprtcResult r = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
  if (r != HIPRTC_SUCCESS) {
    size_t n = 0;
    hiprtcGetProgramLogSize(prog, &n);
    std::string log(n, '\0');
    if (n) hiprtcGetProgramLog(prog, &log[0]);
    hiprtcDestroyProgram(&prog);
    return set_error(HIPNX_EHIP, "fused: compiling a group failed (%s): %.600s", hiprtcGetErrorString(r), log.c_str());
  }
  size_t size = 0;
  hiprtcGetCodeSize(prog, &size);
  std::string code(size, '\0');
  hiprtcGetCode(prog, &code[0]);
  hiprtcDestroyProgram(&prog);
  HIPNX_HIP(hipModuleLoadData(&out->module, code.data()));
  hipError_t e = hipModuleGetFunction(&out->function, out->module, name.c_str());
  if (e == hipSuccess && with_any) e = hipModuleGetFunction(&out->any_length, out->module, any_length(name).c_str());
  if (e != hipSuccess) {
    (void)hipModuleUnload(out->module);
    return hip_fail(e, "hipModuleGetFunction(fused group)");
  }
  return HIPNX_OK;
}

// Makes room in a full table: waits for the stream (a kernel may still be running), then unloads the least
// recently launched quarter.  A program specialised on a constant that changes from call to call (a
// temperature, a learning rate passed as a number) would otherwise grow the table, and the loaded
// modules with it, without bound; each new value still costs one compilation (a few hundred ms).
static int trim_cache(hipnx_ctx *ctx) {
  HIPNX_HIP(hipStreamSynchronize(ctx->stream));
  std::vector<std::pair<uint64_t, const std::string *>> by_age;
  for (auto &kv : ctx->fused_kernels)
    if (!kv.second.in_graph) by_age.emplace_back(kv.second.last_use, &kv.first);
  std::sort(by_age.begin(), by_age.end());
  // (a limit lowered below what is held: down to under the limit)
  const size_t over = ctx->fused_kernels.size() - ctx->fused_cache_max + 1;
  const size_t drop = std::min(by_age.size(), std::max<size_t>(over, ctx->fused_cache_max / 4));
  std::vector<std::string> keys;
  for (size_t i = 0; i < drop; i++) keys.push_back(*by_age[i].second);
  for (const std::string &k : keys) {
    auto it = ctx->fused_kernels.find(k);
    (void)hipModuleUnload(it->second.module);
    ctx->fused_kernels.erase(it);
  }
  return HIPNX_OK;
}

// Launches the compiled kernel for `a`, compiling it first if this context has not seen the program.
// *done = false (and HIPNX_OK) when the caller should run the interpreting kernel instead: the
// program is new and the stream is capturing (compiling and loading a module is no work to record).
// `a` holds what kernels over random words take too, the others are handed the block in front of it.
// `walk`: a group of lanes takes a row, the grid follows from how many; `grid` is the grid otherwise.
int fused_launch_compiled(hipnx_ctx *ctx, const FusedWordsArgs &a, int reduce_op, bool block_per_row, bool walk, int scores_k, unsigned grid, bool *done) {
  *done = false;
  const Keeps keeps = what_is_kept(a, walk);
  int lanes = keeps.tpr;
  const std::string key = make_key(a, keeps, reduce_op, block_per_row, scores_k);
  auto it = ctx->fused_kernels.find(key);
  hipFunction_t function = nullptr;
  if (it == ctx->fused_kernels.end() && ctx->capture) {
    // the program may be there for rows of another length, with a kernel that takes any
    if (a.cols % FE != 0) return HIPNX_OK;
    const size_t same = key.size() - LENGTH_KEY;
    for (it = ctx->fused_kernels.begin(); it != ctx->fused_kernels.end(); ++it)
      if (it->second.any_length && it->first.size() == key.size() && it->first.compare(0, same, key, 0, same) == 0) break;
    if (it == ctx->fused_kernels.end()) return HIPNX_OK;
    function = it->second.any_length;
    lanes = class_lanes(a);
  }
  if (it == ctx->fused_kernels.end()) {
    // a name a profile can tell apart: what the kernel is (a map, a map with its row reduction, stages over rows),
    // how long its program is, and a hash of what it is specialised on
    int stages = 0;
    for (int i = 0; i < a.n_instr; i++) stages += a.ins[i].kind == HIPNX_FUSED_ROW_REDUCE;
    char name[96];
    snprintf(name, sizeof(name), "fused_%s_%dinstr_%08zx", a.words >= 0 ? "words" : a.scores >= 0 ? "scores" : stages ? "stages" : reduce_op != -1 ? "map_reduce" : "map", a.n_instr,
             std::hash<std::string>{}(key) & 0xFFFFFFFFu);
    if (ctx->fused_kernels.size() >= ctx->fused_cache_max)
      if (int st = trim_cache(ctx)) return st;
    hipnx_ctx::FusedKernel k{};
    if (int st = compile(ctx, make_source(a, keeps, reduce_op, block_per_row, scores_k, name), name, has_kernel_for_any_length(a, keeps), &k)) return st;
    if (is_for_any_length(a, keeps)) k.any_length = k.function;
    it = ctx->fused_kernels.emplace(key, k).first;
  }
  if (!function) function = it->second.function;
  it->second.last_use = ++ctx->fused_clock;
  if (ctx->capture) it->second.in_graph = true;  // a recorded launch refers to the loaded module for as long as the graph lives
  // the argument block is the kernel's one by-value parameter: hand it over as the packed buffer it is
  size_t size = a.words >= 0 ? sizeof(FusedWordsArgs) : sizeof(FusedArgs);
  if (walk && a.scores < 0) grid = (unsigned)((a.rows + FBLOCK / lanes - 1) / (FBLOCK / lanes));
  void *config[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, (void *)&a, HIP_LAUNCH_PARAM_BUFFER_SIZE, &size, HIP_LAUNCH_PARAM_END};
  HIPNX_HIP(hipModuleLaunchKernel(function, grid, 1, 1, FBLOCK, 1, 1, 0, ctx->stream, nullptr, config));
  *done = true;
  return HIPNX_OK;
}

}  // namespace hipnx

using namespace hipnx;

extern "C" int hipnx_fused_set_mode(hipnx_ctx *ctx, int mode) {
  Enter in(ctx);
  if (in.status) return in.status;
  if (mode != HIPNX_FUSED_INTERPRETED && mode != HIPNX_FUSED_COMPILED) return set_error(HIPNX_EINVAL, "fused: mode %d", mode);
  ctx->fused_mode = mode;
  return HIPNX_OK;
}

extern "C" int hipnx_fused_set_cache_limit(hipnx_ctx *ctx, int programs) {
  Enter in(ctx);
  if (in.status) return in.status;
  if (programs < 4) return set_error(HIPNX_EINVAL, "fused: a cache limit of %d programs (at least 4)", programs);
  ctx->fused_cache_max = (size_t)programs;
  return HIPNX_OK;
}

extern "C" int hipnx_fused_compiled_count(hipnx_ctx *ctx, int *count) {
  Enter in(ctx);
  if (in.status) return in.status;
  if (!count) return set_error(HIPNX_EINVAL, "fused: null count");
  *count = (int)ctx->fused_kernels.size();
  return HIPNX_OK;
}
