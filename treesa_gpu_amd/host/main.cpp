// main.cpp -- bin/treesa_gpu: the MI355X drop-in for the reference's treesa_gpu binary.
//
// The interface is the reference's: its flags (tsa_cli.cpp), instance / tree / betas files (tsa_host.cpp),
// JSON result keys and trace columns (csrc/treesa_gpu.cu:1896-1920) and exit codes (0 ok, 1 usage, input or
// device error, 2 invalid final tree, 3 failed --check), so treesa_gpu/driver.py runs it through
// TREESA_GPU_BINARY unchanged.  The level loop (csrc/treesa_gpu.cu:1756-1933) is organised here as a
// schedule of levels driven by one of two loops: with independent chains in one energy mode the device
// selects the best chain itself and the host only enqueues; otherwise the host evaluates every selected
// level, keeps the incumbent and runs the population step.  Every device step goes through the C ABI of
// libtreesa_hip.so (include/treesa_hip.h).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "treesa_hip.h"
#include "tsa_cli.h"
#include "tsa_fmt.h"
#include "tsa_host.h"

using namespace tsa;

namespace {

double wall_seconds() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

// An error from the device library; the binary prints it and exits 1.
struct DeviceError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// Page-locked host memory from the library, so that copies of chain records into it run at the link's speed
// (the best record of a 64 x 64 lattice chain is 4 MB).
struct PinnedWords {
  uint64_t* p = nullptr;
  size_t n = 0;
  explicit PinnedWords(size_t words) : n(words) {
    p = static_cast<uint64_t*>(tsa_host_alloc(words * 8));
    if (!p) throw std::bad_alloc();
    std::memset(p, 0, words * 8);
  }
  ~PinnedWords() { tsa_host_free(p); }
  PinnedWords(const PinnedWords&) = delete;
  PinnedWords& operator=(const PinnedWords&) = delete;
};

// One device context (tsa_ctx) with every call checked.
class Device {
 public:
  Device(const tsa_layout_t& lay, const std::vector<uint64_t>& leaf, int leaf_sc, const tsa_config_t& cfg,
         int nchains) {
    create(lay, leaf, leaf_sc, cfg, nchains);
    if (cfg.wide_waves > 0 && describe().compare(0, 3, "lds") == 0) {
      // --wpc plans the wide kernel; where chains sit in LDS it has no effect
      tsa_destroy(ctx_);
      ctx_ = nullptr;
      tsa_config_t automatic = cfg;
      automatic.wide_waves = 0;
      create(lay, leaf, leaf_sc, automatic, nchains);
    }
  }
  ~Device() { tsa_destroy(ctx_); }
  Device(const Device&) = delete;
  Device& operator=(const Device&) = delete;
  tsa_ctx* get() const { return ctx_; }
  void ok(int rc) const {
    if (rc != TSA_OK) throw DeviceError(std::string("treesa_hip: ") + tsa_last_error(ctx_));
  }
  std::string describe() const {
    char b[256] = {0};
    tsa_describe(ctx_, b, sizeof b);
    return b;
  }
  double take_kernel_ms() const {
    double ms = 0;
    ok(tsa_sweeps_ms(ctx_, &ms));
    return ms;
  }
  void counters(uint64_t st[7], uint64_t chunks[2]) const {
    ok(tsa_stats(ctx_, st));
    ok(tsa_chunk_stats(ctx_, chunks));
  }

 private:
  void create(const tsa_layout_t& lay, const std::vector<uint64_t>& leaf, int leaf_sc, const tsa_config_t& cfg,
              int nchains) {
    if (tsa_create(&lay, leaf.data(), leaf_sc, &cfg, nchains, &ctx_) == TSA_OK) return;
    const std::string msg = tsa_last_error(nullptr);
    if (msg.find("fit") != std::string::npos)
      throw DeviceError("chains do not fit in shared memory (try --kernel warp / --lpc 32)");
    throw DeviceError("treesa_hip: " + msg);
  }
  tsa_ctx* ctx_ = nullptr;
};

// One β level of the schedule: its inverse temperature, energy mode and sweeps.
struct Level {
  float beta;
  int mode;
  int niters;
};

// A chain's energies at an evaluated level.
struct Energies {
  std::vector<float> lc;
  std::vector<int32_t> sc, ns;
  explicit Energies(int n) : lc(n), sc(n), ns(n) {}
};

// Small JSON writer: keys in insertion order, numbers in the reference's printed precision.
class Json {
 public:
  void key(const char* k) {
    out_ += first_ ? "{\"" : ",\n \"";
    out_ += k;
    out_ += "\": ";
    first_ = false;
  }
  void fixed6(const char* k, double v) { put(k, "%.6f", v); }
  // times in seconds: %.6e, non-finite values as null (csrc/treesa_gpu.cu:70-76)
  void sci6(const char* k, double v) {
    if (std::isfinite(v)) put(k, "%.6e", v);
    else raw(k, "null");
  }
  // a double that reads back to the same bits (%.17g), non-finite values as null
  void exact(const char* k, double v) {
    if (std::isfinite(v)) put(k, "%.17g", v);
    else raw(k, "null");
  }
  void integer(const char* k, long long v) { put(k, "%lld", v); }
  void boolean(const char* k, bool v) { raw(k, v ? "true" : "false"); }
  void text(const char* k, const std::string& v) { raw(k, "\"" + v + "\""); }
  void raw(const char* k, const std::string& v) {
    key(k);
    out_ += v;
  }
  std::string finish() { return out_ + "}\n"; }

 private:
  template <typename T>
  void put(const char* k, const char* fmt, T v) {
    char b[64];
    snprintf(b, sizeof b, fmt, v);
    raw(k, b);
  }
  std::string out_;
  bool first_ = true;
};

// The integer after `key` in a kernel description (tsa_describe), or dflt.
int desc_int(const std::string& desc, const char* key, int dflt) {
  const size_t p = desc.find(key);
  return p == std::string::npos ? dflt : atoi(desc.c_str() + p + strlen(key));
}

// Widths as the reference reports them (32-bit words): its register template width (0 on the wide path) and
// its words per label set (csrc/treesa_gpu.cu:1439, 2078-2085).
void reference_widths(int nlab, bool wide, int* W32, int* nw32) {
  const int w = (nlab + 31) / 32;
  if (wide || w > 16) {
    *W32 = 0;
    *nw32 = (w + 3) & ~3;
    return;
  }
  *W32 = w <= 1 ? 1 : w <= 2 ? 2 : w <= 4 ? 4 : w <= 8 ? 8 : w <= 12 ? 12 : 16;
  *nw32 = *W32;
}

class Run {
 public:
  Run(const Network& N, const Options& O) : N_(N), O_(O) {
    if (tsa_layout(N.m, N.nlab, O.wide ? 1 : 0, &lay_) != TSA_OK) throw DeviceError(tsa_last_error(nullptr));
    geo_ = Geometry{lay_.W, lay_.ch_off, lay_.s_off, lay_.chain_words};
    leaf_ = leaf_sets(N, lay_.W);
    model_ = model_log2(O.model);
    resolve_kernel();
    fill_config();
  }
  int anneal();
  int check();

 private:
  const Network& N_;
  const Options& O_;
  tsa_layout_t lay_{};
  Geometry geo_{};
  tsa_config_t cfg_{};
  std::vector<uint64_t> leaf_;
  ModelLog2 model_{};
  std::string kernel_;  // the reference's kernel name after its automatic choice
  int order_ = TSA_ORDER_PAR;
  std::unique_ptr<Device> dev_;
  // start trees (built once)
  std::vector<std::vector<uint32_t>> trees_;
  std::vector<double> init_tcs_;
  double t_trees_ = 0;
  bool have_trees_ = false;
  // level loop state
  std::vector<Level> sched_;
  int mode_ = 0;
  double kernel_ms_ = 0;
  std::string trace_;
  FILE* level_log_ = nullptr;

  void resolve_kernel();
  void fill_config();
  const std::vector<std::vector<uint32_t>>& start_trees();
  std::vector<uint64_t> start_population();
  void build_schedule();
  Scoring scoring(int mode) const {
    Scoring S;
    S.mode = mode;
    S.slicing = O_.slicing;
    S.select_sc = O_.select_sc;
    S.sc_target = O_.sc_target;
    S.sc_weight = O_.sc_weight;
    return S;
  }
  tsa_select_t device_scoring() const {
    tsa_select_t s{};
    s.mode = O_.mode;
    s.slicing = O_.slicing ? 1 : 0;
    s.select_sc = O_.select_sc ? 1 : 0;
    s.sc_target = O_.sc_target;
    s.sc_weight = O_.sc_weight;
    return s;
  }
  bool evaluated_level(int lev) const {
    const int n = (int)sched_.size();
    const bool last = lev + 1 == n;
    return last || lev % O_.eval_every == O_.eval_every - 1 || sched_[lev + 1].mode != sched_[lev].mode;
  }
  const uint32_t* children(const uint64_t* rec) const { return reinterpret_cast<const uint32_t*>(rec + lay_.ch_off); }
  const uint64_t* slices(const uint64_t* rec) const { return O_.slicing ? rec + lay_.s_off : nullptr; }
  void add_trace(double t, int lev, float lc, int sc, double meanE, int families, int ns, double meanNs);
  void progress(int lev, float lc, int sc, int ns, double meanE, double meanNs, int families, double t) const;
  void warm_up(const std::vector<uint64_t>& pop, uint64_t st0[7], uint64_t ch0[2]);
  bool anneal_on_device();
  int loop_on_device(PinnedWords& best, double t0);
  int loop_on_host(PinnedWords& best, double t0, HostEnergy& h1, bool& staged, int& nresample);
  std::string kernel_label() const;
};

void Run::resolve_kernel() {
  if (O_.order != "par" && O_.order != "preorder") throw InputError("--order par|preorder");
  // par order runs the par kernel; an explicit --kernel other than auto / par, or lanes per chain other than
  // 32, means the pre-order sweep (csrc/treesa_gpu.cu:1480-1483)
  kernel_ = O_.kernel;
  if (kernel_ == "auto" && O_.order == "par" && O_.lpc == 32) kernel_ = "par";
  static const char* known[] = {"auto", "par", "seq", "seqsm", "warp", "warpsm", "block"};
  if (std::none_of(std::begin(known), std::end(known), [&](const char* k) { return kernel_ == k; }))
    throw InputError("unknown --kernel " + kernel_);
  order_ = kernel_ == "par" ? TSA_ORDER_PAR : TSA_ORDER_PREORDER;
  if (O_.par_band == 1 || O_.par_band > 16 || O_.par_band < 0) throw InputError("--par-band L: 0 (off) or 2..16");
  const bool moves = O_.slicing && O_.random_slices == 0 && O_.slice_moves > 0;
  if (moves && (kernel_ == "seq" || kernel_ == "seqsm" || O_.lpc != 32))
    throw InputError("slice moves need the warp kernels with --lpc 32");
  if (O_.nchains < 1) throw InputError("--nchains must be at least 1");
  if (O_.eval_every < 1) throw InputError("--eval-every must be at least 1");
  if (O_.level_blocks < 0 || O_.level_blocks > 8) throw InputError("--level-blocks K: 0 (automatic) or 1..8");
  if (O_.scheme != "indep" && O_.scheme != "pa" && O_.scheme != "trunc") throw InputError("--scheme indep|pa|trunc");
}

void Run::fill_config() {
  std::memset(&cfg_, 0, sizeof cfg_);
  mode_ = O_.mode;
  cfg_.mode = O_.mode;
  cfg_.sc_target = (float)O_.sc_target;
  cfg_.sc_weight = (float)O_.sc_weight;
  const uint64_t key = splitmix64(O_.seed);  // Philox key (csrc/treesa_gpu.cu:1457-1459)
  cfg_.key0 = (uint32_t)key;
  cfg_.key1 = (uint32_t)(key >> 32);
  cfg_.slicing = O_.slicing ? 1 : 0;
  cfg_.slice_moves = (O_.slicing && O_.random_slices == 0) ? O_.slice_moves : 0;
  cfg_.slice_every = std::max(1, O_.slice_every);
  cfg_.max_slices = O_.max_slices > 0 ? O_.max_slices : N_.nlab;
  cfg_.par_follow = O_.par_follow;
  cfg_.par_band = O_.par_band;
  cfg_.kernel = (kernel_ == "warpsm" || kernel_ == "seqsm")                       ? TSA_KERNEL_LDS
                : (kernel_ == "warp" || kernel_ == "seq" || kernel_ == "block") ? TSA_KERNEL_GLOBAL
                                                                                : TSA_KERNEL_AUTO;
  cfg_.lpeak = model_.lpeak;
  cfg_.lbw = model_.lbw;
  cfg_.llaunch = model_.llaunch;
  cfg_.m0 = model_.m0;
  cfg_.n0 = model_.n0;
  cfg_.k0 = model_.k0;
  cfg_.v2_l3launch = model_.v2_l3launch;
  cfg_.v2_lperm2 = model_.v2_lperm2;
  cfg_.v2_lcc_bit = model_.v2_lcc_bit;
  cfg_.v2_lcc_cell = model_.v2_lcc_cell;
  cfg_.v2_ltc_bit = model_.v2_ltc_bit;
  cfg_.v2_ltc_pad = model_.v2_ltc_pad;
  cfg_.v2_ltc_out = model_.v2_ltc_out;
  cfg_.v2_lsmall_cell = model_.v2_lsmall_cell;
  cfg_.v2_small_rank = model_.v2_small_rank;
  cfg_.wide_waves = O_.wpc > 0 ? (O_.wpc + 1) / 2 : 0;  // --wpc counts 32-lane warps
  cfg_.wide_wgs = O_.wide_wgs;
  cfg_.wide_lanes = O_.wide_lanes;
  cfg_.fused_energy = O_.eval_every == 1 ? 1 : 0;  // every level evaluated: the sweep kernel evaluates too
  cfg_.sums = O_.no_sum ? -1 : (O_.force_sum ? 1 : 0);
  cfg_.track_overlap = O_.no_overlap ? -1 : 0;
  cfg_.draw_waves = O_.draw_waves;
  cfg_.level_loop = O_.level_loop ? 1 : 0;
  cfg_.level_blocks = O_.level_blocks;
}

const std::vector<std::vector<uint32_t>>& Run::start_trees() {
  if (have_trees_) return trees_;
  const double t = wall_seconds();
  if (!O_.tree_file.empty()) {
    trees_ = read_tree_file(O_.tree_file, N_.m);
  } else if (O_.init == "spectral") {
    for (const SpectralOrder& so : spectral_orders(N_, std::max(1, O_.spectral_k), 24, 24, O_.seed)) {
      trees_.push_back(path_tree(so.order));
      init_tcs_.push_back(so.tc);
    }
  } else if (O_.init == "greedy") {
    double tc = 0;
    trees_.push_back(greedy_tree(N_, std::max(1, O_.greedy_repeat), O_.seed, &tc));
    init_tcs_.push_back(tc);
  }
  t_trees_ = wall_seconds() - t;
  have_trees_ = true;
  return trees_;
}

std::vector<uint64_t> Run::start_population() {
  std::vector<uint64_t> S0(lay_.W, 0ull);
  for (size_t p = 0; p < O_.init_slices.size();) {
    char* e = nullptr;
    const long l = strtol(O_.init_slices.c_str() + p, &e, 10);
    const size_t q = (size_t)(e - O_.init_slices.c_str());
    if (q == p) break;
    if (l < 0 || l >= N_.nlab) throw InputError("bad --init-slices label");
    S0[l >> 6] |= 1ull << (l & 63);
    p = q;
    while (p < O_.init_slices.size() && (O_.init_slices[p] == ',' || O_.init_slices[p] == ' ')) p++;
  }
  std::vector<uint64_t> pop;
  build_population(N_, geo_, start_trees(), O_.nchains, O_.seed, S0, O_.random_slices, pop);
  return pop;
}

void Run::build_schedule() {
  std::vector<float> b = parse_schedule(O_.betas);
  if (O_.max_levels > 0 && (int)b.size() > O_.max_levels) b.resize(O_.max_levels);
  sched_.clear();
  for (float x : b) sched_.push_back({x, O_.mode, O_.niters});
  if (!O_.stage2_betas.empty())
    for (float x : parse_schedule(O_.stage2_betas))
      sched_.push_back({x, O_.stage2_mode, O_.stage2_niters > 0 ? O_.stage2_niters : O_.niters});
}

// One trace row, the characters of "%s[%.4f,%d,%.4f,%.6f,%d,%.6f,%d,%d,%d,%.3f]" (tsa_fmt.h)
void Run::add_trace(double t, int lev, float lc, int sc, double meanE, int families, int ns, double meanNs) {
  char b[1600];
  int n = 0;
  if (!trace_.empty()) b[n++] = ',';
  b[n++] = '[';
  n += fmt_fixed(b + n, t, 4);
  b[n++] = ',';
  n += fmt_int(b + n, lev);
  b[n++] = ',';
  n += fmt_fixed(b + n, (double)sched_[lev].beta, 4);
  b[n++] = ',';
  n += fmt_fixed(b + n, (double)lc, 6);
  b[n++] = ',';
  n += fmt_int(b + n, sc);
  b[n++] = ',';
  n += fmt_fixed(b + n, meanE, 6);
  for (int v : {families, mode_, ns}) {
    b[n++] = ',';
    n += fmt_int(b + n, v);
  }
  b[n++] = ',';
  n += fmt_fixed(b + n, meanNs, 3);
  b[n++] = ']';
  trace_.append(b, (size_t)n);
}

void Run::progress(int lev, float lc, int sc, int ns, double meanE, double meanNs, int families, double t) const {
  if (O_.quiet || !(lev % 25 == 0 || lev + 1 == (int)sched_.size())) return;
  fprintf(stderr, "[level %d/%zu] beta %.3f | best: lcost %.3f sc %d |S| %d | mean E %.3f mean |S| %.2f | families %d | %.2f s\n",
          lev, sched_.size(), (double)sched_[lev].beta, (double)lc, sc, ns, meanE, meanNs, families, t);
}

// Untimed levels before the timed loop (clocks up, code objects loaded, the tracking buffers and the second
// stream used once; for the host-side loop a resampling and an asynchronous record copy), then the start
// population again; the counters are read so that the run reports only the timed levels.
void Run::warm_up(const std::vector<uint64_t>& pop, uint64_t st0[7], uint64_t ch0[2]) {
  tsa_ctx* c = dev_->get();
  const int n = (int)sched_.size();
  const bool track = O_.scheme == "indep" && O_.stage2_betas.empty() && !O_.host_select;
  Energies e(O_.nchains);
  if (track) {
    const tsa_select_t s = device_scoring();
    dev_->ok(tsa_track_begin(c, &s, n));
    // the level loop in one launch: one whole untimed schedule (its kernel and buffers are the timed loop's)
    if (O_.bench_warmup > 0 && anneal_on_device()) {
      std::vector<uint64_t> rec(lay_.chain_words);
      std::vector<tsa_trace_row_t> rows(n);
      int32_t bc, bl;
      double bs, hz;
      uint64_t tk;
      dev_->ok(tsa_track_end(c, &bc, &bl, &bs, rec.data(), rows.data(), &tk, &hz));
      (void)dev_->take_kernel_ms();
      dev_->ok(tsa_upload(c, pop.data()));
      dev_->counters(st0, ch0);
      return;
    }
  }
  for (int k = 0; k < O_.bench_warmup; k++) {
    const Level& L = sched_[k % n];
    dev_->ok(tsa_sweeps(c, order_, L.beta, (uint32_t)k, L.niters));
    if (track) dev_->ok(tsa_track(c, k % n));
    dev_->ok(tsa_energy(c, e.lc.data(), e.sc.data(), e.ns.data()));
  }
  if (!track && O_.bench_warmup > 0) {
    // the host-side loop's other device work used once before the clock starts (a kernel's first launch loads
    // its code object): a resampling with identity ancestors and a record copied behind the device's work
    std::vector<int> same(O_.nchains);
    for (int k = 0; k < O_.nchains; k++) same[k] = k;
    dev_->ok(tsa_resample(c, same.data()));
    PinnedWords rec(lay_.chain_words);
    dev_->ok(tsa_download_async(c, 0, 1, rec.p));
    dev_->ok(tsa_wait(c));
  }
  if (track) {
    std::vector<uint64_t> rec(lay_.chain_words);
    std::vector<tsa_trace_row_t> rows(n);
    int32_t bc, bl;
    double bs, hz;
    uint64_t tk;
    dev_->ok(tsa_track_end(c, &bc, &bl, &bs, rec.data(), rows.data(), &tk, &hz));
  }
  (void)dev_->take_kernel_ms();
  dev_->ok(tsa_upload(c, pop.data()));
  dev_->counters(st0, ch0);
}

// The whole schedule through tsa_anneal (one launch where every chain is resident at once, else the library's
// per-level launches), after tsa_track_begin; false with --level-launches or a level of no sweep.
bool Run::anneal_on_device() {
  const int n = (int)sched_.size();
  if (O_.level_launches) return false;
  std::vector<float> betas(n);
  std::vector<int32_t> niters(n);
  std::vector<uint8_t> ev(n);
  for (int lev = 0; lev < n; lev++) {
    if (sched_[lev].niters < 1) return false;
    betas[lev] = sched_[lev].beta;
    niters[lev] = sched_[lev].niters;
    ev[lev] = evaluated_level(lev) ? 1 : 0;
  }
  dev_->ok(tsa_anneal(dev_->get(), order_, 0, n, betas.data(), niters.data(), ev.data(), 0u));
  return true;
}

// Independent chains in one energy mode: the whole schedule through tsa_anneal, or (--level-launches) every
// level's sweeps and, at evaluated levels, the device's own energy and selection kernels, enqueued; the host
// waits once, at the end.  The selection is the reference's (lowest score, first
// chain and first level on ties); the trace's time column comes from the device clock, scaled to the host's
// wall time of the loop.
int Run::loop_on_device(PinnedWords& best, double t0) {
  tsa_ctx* c = dev_->get();
  const int n = (int)sched_.size();
  const tsa_select_t s = device_scoring();
  dev_->ok(tsa_track_begin(c, &s, n));
  std::vector<char> evaluated(n, 0);
  for (int lev = 0; lev < n; lev++) evaluated[lev] = evaluated_level(lev) ? 1 : 0;
  if (!anneal_on_device()) {
    uint32_t sweep = 0;
    for (int lev = 0; lev < n; lev++) {
      dev_->ok(tsa_sweeps(c, order_, sched_[lev].beta, sweep, sched_[lev].niters));
      sweep += (uint32_t)sched_[lev].niters;
      if (evaluated[lev]) dev_->ok(tsa_track(c, lev));
    }
  }
  // the best and the trace rows first: their copies are enqueued behind the device's work while it still runs,
  // and the call returns when it ends; the kernel time after that finds every timing event complete
  std::vector<tsa_trace_row_t> rows(n);
  int32_t best_chain = -1, best_level = -1;
  double best_score = 0, hz = 1;
  uint64_t tk0 = 0;
  dev_->ok(tsa_track_end(c, &best_chain, &best_level, &best_score, best.p, rows.data(), &tk0, &hz));
  const double wall = wall_seconds() - t0;
  kernel_ms_ += dev_->take_kernel_ms();
  const double span = std::max(1.0, (double)(rows[n - 1].ticks - tk0));
  for (int lev = 0; lev < n; lev++) {
    if (!evaluated[lev]) continue;
    const tsa_trace_row_t& r = rows[lev];
    const double t = wall * (double)(r.ticks - tk0) / span;
    add_trace(t, lev, r.lc, r.sc, r.meanE, O_.nchains, r.ns, r.meanNs);
    progress(lev, r.lc, r.sc, r.ns, r.meanE, r.meanNs, O_.nchains, t);
    if (level_log_) {
      uint32_t bits;
      std::memcpy(&bits, &r.lc, 4);
      fprintf(level_log_,
              "{\"level\": %d, \"best\": %d, \"score\": %.17g, \"lc_bits\": %u, \"sc\": %d, \"ns\": %d, "
              "\"families\": %d, \"meanE\": %.17g, \"resampled\": false}\n",
              lev, r.chain, r.score, bits, r.sc, r.ns, O_.nchains, r.meanE);
    }
  }
  return best_chain;
}

// The host-side loop (population schemes, two-stage runs, --host-select): at every evaluated level the host
// reads every chain's energies, selects, writes the trace row and, between levels of one energy mode, runs the
// population step.
int Run::loop_on_host(PinnedWords& best, double t0, HostEnergy& h1, bool& staged, int& nresample) {
  tsa_ctx* c = dev_->get();
  const int n = (int)sched_.size(), nc = O_.nchains;
  Energies e(nc);
  std::vector<double> E(nc);
  std::vector<int> family(nc), mark(nc);
  for (int k = 0; k < nc; k++) family[k] = k;
  std::mt19937_64 pa_rng(splitmix64(O_.seed + 777));  // the uniforms of systematic resampling
  float beta_resampled = n > 0 ? sched_[0].beta : 0.f;  // β of the population's last reweighting
  double incumbent = INFINITY;
  int best_chain = -1;
  uint32_t sweep = 0;
  bool enqueued = false;  // this level's sweeps were enqueued at the end of the previous level
  for (int lev = 0; lev < n; lev++) {
    const Level& L = sched_[lev];
    if (L.mode != mode_) {
      // stage switch: the stage-1 incumbent stays, scored in the new energy by its host double energy (its
      // record arrives with the copies enqueued so far)
      dev_->ok(tsa_wait(c));
      h1 = host_energy(N_, lay_.W, model_, best.p, children(best.p), leaf_, slices(best.p));
      staged = true;
      mode_ = L.mode;
      dev_->ok(tsa_set_mode(c, mode_));
      incumbent = selection_score(scoring(mode_), (float)std::log2(mode_ == 1 ? h1.time : h1.time2), h1.sc, h1.ns);
      beta_resampled = L.beta;
    }
    if (!enqueued) dev_->ok(tsa_sweeps(c, order_, L.beta, sweep, L.niters));
    enqueued = false;
    sweep += (uint32_t)L.niters;
    if (!evaluated_level(lev)) continue;
    dev_->ok(tsa_energy(c, e.lc.data(), e.sc.data(), e.ns.data()));
    kernel_ms_ += dev_->take_kernel_ms();
    const Scoring S = scoring(mode_);
    int bi = 0;
    double bs = INFINITY, sumE = 0, sumNs = 0;
    for (int k = 0; k < nc; k++) {
      const double s = selection_score(S, e.lc[k], e.sc[k], e.ns[k]);
      if (s < bs) {
        bs = s;
        bi = k;
      }
      E[k] = population_energy(S, e.lc[k], e.sc[k], e.ns[k]);
      sumE += E[k];
      sumNs += e.ns[k];
    }
    if (bs < incumbent) {  // the record as it is now, copied behind the device's work
      incumbent = bs;
      best_chain = bi;
      dev_->ok(tsa_download_async(c, bi, 1, best.p));
    }
    // population step, not at the last level nor across an energy change
    const bool last = lev + 1 == n;
    const bool next_same = !last && sched_[lev + 1].mode == mode_;
    std::vector<int> anc;
    if (next_same) {
      if (O_.scheme == "pa") {
        const double db = (double)(sched_[lev + 1].beta - beta_resampled);  // a float difference, as the reference
        beta_resampled = sched_[lev + 1].beta;
        const double u = std::uniform_real_distribution<double>(0, 1)(pa_rng);
        anc = systematic_ancestors(E, db, u);
      } else if (O_.scheme == "trunc") {
        anc = truncation_ancestors(E, O_.trunc_frac);
      }
    }
    if (!anc.empty()) dev_->ok(tsa_resample(c, anc.data()));
    // the next level's sweeps go to the device before this level's bookkeeping (not across an energy change,
    // whose incumbent needs the host first)
    if (next_same) {
      dev_->ok(tsa_sweeps(c, order_, sched_[lev + 1].beta, sweep, sched_[lev + 1].niters));
      enqueued = true;
    }
    std::fill(mark.begin(), mark.end(), 0);
    int families = 0;
    for (int k = 0; k < nc; k++) families += mark[family[k]]++ == 0;
    const double t = wall_seconds() - t0;
    add_trace(t, lev, e.lc[bi], e.sc[bi], sumE / nc, families, e.ns[bi], sumNs / nc);
    progress(lev, e.lc[bi], e.sc[bi], e.ns[bi], sumE / nc, sumNs / nc, families, t);
    if (level_log_) {
      uint32_t bits;
      std::memcpy(&bits, &e.lc[bi], 4);
      fprintf(level_log_,
              "{\"level\": %d, \"best\": %d, \"score\": %.17g, \"lc_bits\": %u, \"sc\": %d, \"ns\": %d, "
              "\"families\": %d, \"meanE\": %.17g, \"resampled\": %s",
              lev, bi, bs, bits, e.sc[bi], e.ns[bi], families, sumE / nc, anc.empty() ? "false" : "true");
      if (!anc.empty()) {
        fprintf(level_log_, ", \"anc\": [");
        for (int k = 0; k < nc; k++) fprintf(level_log_, "%s%d", k ? "," : "", anc[k]);
        fprintf(level_log_, "]");
      }
      fprintf(level_log_, "}\n");
    }
    if (!anc.empty()) {
      std::vector<int> f2(nc);
      for (int k = 0; k < nc; k++) f2[k] = family[anc[k]];
      family.swap(f2);
      nresample++;
    }
  }
  dev_->ok(tsa_wait(c));  // the best record's last copy
  kernel_ms_ += dev_->take_kernel_ms();
  return best_chain;
}

std::string Run::kernel_label() const {
  if (order_ == TSA_ORDER_PAR) return "par";
  return dev_->describe().compare(0, 3, "lds") == 0 ? "warpsm" : "warp";
}

int Run::anneal() {
  build_schedule();
  if (sched_.empty()) throw InputError("no levels (empty --betas)");
  const double t_start = wall_seconds();
  const std::vector<uint64_t> pop = start_population();  // input errors surface before the device is touched
  dev_ = std::make_unique<Device>(lay_, leaf_, N_.largest_tensor(), cfg_, O_.nchains);
  tsa_ctx* c = dev_->get();
  dev_->ok(tsa_upload(c, pop.data()));
  uint64_t st0[7] = {0, 0, 0, 0, 0, 0, 0}, ch0[2] = {0, 0};
  if (O_.bench_warmup > 0) warm_up(pop, st0, ch0);
  if (!O_.level_log.empty()) {
    level_log_ = fopen(O_.level_log.c_str(), "w");
    if (!level_log_) throw InputError("cannot open " + O_.level_log);
  }
  PinnedWords best(lay_.chain_words);  // allocated (its pages touched) before the clock starts
  const double t_init = wall_seconds() - t_start;
  const double t0 = wall_seconds();
  HostEnergy h1;
  bool staged = false;
  int nresample = 0;
  const bool on_device = O_.scheme == "indep" && O_.stage2_betas.empty() && !O_.host_select;
  const int best_chain = on_device ? loop_on_device(best, t0) : loop_on_host(best, t0, h1, staged, nresample);
  const double t_anneal = wall_seconds() - t0;
  if (level_log_) fclose(level_log_);
  if (!O_.dump_population.empty()) {
    // the final population as the level loop left it (nchains records of chain_words words, in chain order)
    std::vector<uint64_t> all((size_t)O_.nchains * lay_.chain_words);
    dev_->ok(tsa_download(c, 0, O_.nchains, all.data()));
    FILE* f = fopen(O_.dump_population.c_str(), "wb");
    if (!f || fwrite(all.data(), 8, all.size(), f) != all.size()) {
      if (f) fclose(f);
      throw InputError("cannot write " + O_.dump_population);
    }
    fclose(f);
  }
  uint32_t total_sweeps = 0;
  for (const Level& L : sched_) total_sweeps += (uint32_t)L.niters;
  uint64_t st[7], chunks[2];
  dev_->counters(st, chunks);
  for (int k = 0; k < 7; k++) st[k] -= st0[k];
  for (int k = 0; k < 2; k++) chunks[k] -= ch0[k];

  // the final tree, verified from scratch: its label sets from the topology must equal the maintained ones
  // (the device-side loop returns only the tree; then the chain's live record is checked instead)
  const uint32_t* bch = children(best.p);
  std::vector<uint64_t> lab((size_t)lay_.nint * lay_.W, 0ull);
  const bool valid = topology_labels(N_, lay_.W, bch, lab.data());
  bool labels_ok = valid && std::equal(lab.begin(), lab.end(), best.p);
  if (on_device && best_chain >= 0) {
    std::vector<uint64_t> live(lay_.chain_words), lab2((size_t)lay_.nint * lay_.W, 0ull);
    dev_->ok(tsa_download(c, best_chain, 1, live.data()));
    labels_ok = valid && topology_labels(N_, lay_.W, children(live.data()), lab2.data()) &&
                std::equal(lab2.begin(), lab2.end(), live.begin());
    std::copy(lab.begin(), lab.end(), best.p);
  }
  int n_repair = 0;
  if (O_.slicing && valid) n_repair = greedy_repair(N_, lay_.W, lab.data(), leaf_, best.p + lay_.s_off, O_.sc_target);
  const HostEnergy HE = host_energy(N_, lay_.W, model_, lab.data(), bch, leaf_, slices(best.p));
  const double ks = kernel_ms_ / 1e3;
  if (!O_.quiet)
    fprintf(stderr,
            "best: tc %.4f sc %d |S| %d (+%d repaired), gpu model %.4e s, h100 model %.4e s per slice\n"
            "time: anneal %.3f s, set-up %.3f s, sweep kernels %.3f s: %.3e proposals/s, %.3e node visits/s; "
            "slice moves %llu of %llu accepted\n",
            HE.tc, HE.sc, HE.ns, n_repair, HE.time, HE.time2, t_anneal, t_init, ks, ks > 0 ? st[0] / ks : 0.0,
            ks > 0 ? (double)total_sweeps * O_.nchains * (N_.m - 1) / ks : 0.0, (unsigned long long)st[5],
            (unsigned long long)st[4]);

  const std::string desc = dev_->describe();
  const size_t sp = desc.find(" sums=");
  const int nsum = (sp != std::string::npos && atoi(desc.c_str() + sp + 6) > 0) ? (lay_.W / 2 + 31) / 32 : 0;
  int W32 = 0, nw32 = 0;
  reference_widths(N_.nlab, lay_.runtime_width != 0, &W32, &nw32);
  std::string sliced = "[";
  for (int l = 0; l < N_.nlab && O_.slicing; l++)
    if (best.p[lay_.s_off + (l >> 6)] >> (l & 63) & 1u) sliced += (sliced.size() > 1 ? "," : "") + std::to_string(l);
  sliced += "]";
  std::string tree = "[";
  for (int i = 0; i < lay_.nint; i++)
    tree += (i ? ",[" : "[") + std::to_string(bch[i] & 0xFFFFu) + "," + std::to_string(bch[i] >> 16) + "]";
  tree += "]";

  Json j;
  j.fixed6("tc", HE.tc);
  j.exact("tc_exact", HE.tc);
  j.integer("sc", HE.sc);
  j.sci6("gpu_time", HE.time);
  j.sci6("h100_time", HE.time2);
  j.boolean("valid", valid);
  j.boolean("labels_ok", labels_ok);
  j.integer("best_chain", best_chain);
  j.boolean("slicing", O_.slicing);
  j.integer("nsliced", HE.ns);
  j.integer("n_repair", n_repair);
  j.fixed6("tc_total", HE.tc + HE.ns);
  j.sci6("gpu_time_total", HE.time * std::exp2((double)HE.ns));
  j.sci6("h100_time_total", HE.time2 * std::exp2((double)HE.ns));
  j.raw("sliced", sliced);
  j.fixed6("t_anneal", t_anneal);
  j.fixed6("t_init", t_init);
  j.fixed6("kernel_s", ks);
  static const char* counter_keys[7] = {"proposals",       "accepts",       "warp_steps", "node_visits",
                                        "slice_proposals", "slice_accepts", "busy_lanes"};
  for (int k = 0; k < 7; k++) j.integer(counter_keys[k], (long long)st[k]);
  // the visit mapping of the last sweeps in the reference's terms: lanes per proposal (coop_*), waves that visit for a
  // chain (wpc) and the proposals one of their rounds holds (lpc: waves x 64 / lanes in par order, a step's 64 nodes in
  // pre-order).  warp_steps counts what the reference's kernels count (csrc/treesa_gpu.cu:716, 990): rounds of
  // up to lpc visits in pre-order, phases in par order; so node_visits / (lpc * warp_steps) is the lane
  // occupancy of a pre-order sweep and the visits per phase and visit slot of a par sweep, as there
  // (bench/throughput.py:68).
  const bool wide = desc.compare(0, 5, "wide ") == 0 && desc.find(" sweeps=one_lane") == std::string::npos;
  const bool par = order_ == TSA_ORDER_PAR;
  const int G = !par ? desc_int(desc, " preorder_lanes=", 1) : desc_int(desc, wide ? " G=" : " team_lanes=", 1);
  const int wpc = !par   ? desc_int(desc, " preorder_waves=", 1)
                  : wide ? desc_int(desc, " waves/block=", 1) * desc_int(desc, " blocks/chain=", 1)
                         : desc_int(desc, " par_team_waves=", 1);
  j.integer("coop_max", G);
  j.integer("coop_min", G);
  j.integer("coop_full", G);
  j.integer("par_follow", O_.par_follow);
  j.integer("par_band", O_.par_band);
  j.integer("nsum", nsum);
  j.integer("wpc", wpc);
  j.text("order", order_ == TSA_ORDER_PAR ? "par" : "preorder");
  j.integer("nchains", O_.nchains);
  j.integer("niters", O_.niters);
  j.integer("nlevels", (long long)sched_.size());
  j.integer("total_sweeps", total_sweeps);
  j.integer("W", W32);
  j.integer("nw", nw32);
  j.integer("W64", lay_.W);
  j.integer("word_bits", 64);
  j.integer("lpc", par ? wpc * 64 / G : 64);
  j.text("kernel", kernel_label());
  j.text("hip_kernel", desc);
  j.text("scheme", O_.scheme);
  j.integer("mode", O_.mode);
  j.integer("nresample", nresample);
  j.integer("sum_chunks", (long long)chunks[0]);
  j.integer("sum_xchunks", (long long)chunks[1]);
  if (!init_tcs_.empty()) {
    j.text("init", O_.init);
    j.fixed6("t_start_trees", t_trees_);
    std::string v = "[";
    for (size_t i = 0; i < init_tcs_.size(); i++) {
      char b[32];
      snprintf(b, sizeof b, "%s%.4f", i ? ", " : "", init_tcs_[i]);
      v += b;
    }
    j.raw("init_tcs", v + "]");
  }
  if (staged) {
    j.fixed6("stage1_tc", h1.tc);
    j.exact("stage1_tc_exact", h1.tc);
    j.integer("stage1_sc", h1.sc);
    j.integer("stage1_nsliced", h1.ns);
    j.sci6("stage1_gpu_time", h1.time);
    j.sci6("stage1_h100_time", h1.time2);
    j.sci6("stage1_h100_time_total", h1.time2 * std::exp2((double)h1.ns));
  }
  j.raw("trace_cols",
        "[\"t\", \"level\", \"beta\", \"best_lcost_per_slice\", \"best_sc\", \"mean_E\", \"families\", \"mode\", "
        "\"best_nsliced\", \"mean_nsliced\"]");
  j.raw("trace", "[" + trace_ + "]");
  j.raw("tree", tree);
  const std::string text = j.finish();
  FILE* f = O_.out_file.empty() ? stdout : fopen(O_.out_file.c_str(), "w");
  if (!f) throw InputError("cannot open " + O_.out_file);
  fputs(text.c_str(), f);
  if (f != stdout) fclose(f);
  return valid && labels_ok ? 0 : 2;
}

// --check (csrc/treesa_gpu.cu:1940-2061): sweeps of every level, then [1] every chain is a valid tree whose
// label sets equal its topology's, [2] the energy kernel agrees with the host double computation, [3] the
// other kernel mapping (chain in LDS or wide vs one wave in HBM) is bit-identical.  The CPU-reference
// comparison [4] needs the oracle, which this binary does not link; the test suite runs it through the C ABI.
int Run::check() {
  build_schedule();
  sched_.resize(std::min(sched_.size(), parse_schedule(O_.betas).size()));  // stage 1 only
  const std::vector<uint64_t> init = start_population();
  dev_ = std::make_unique<Device>(lay_, leaf_, N_.largest_tensor(), cfg_, O_.nchains);
  tsa_ctx* c = dev_->get();
  auto sweep_all = [&](tsa_ctx* x) {
    for (size_t lev = 0; lev < sched_.size(); lev++)
      dev_->ok(tsa_sweeps(x, order_, sched_[lev].beta, (uint32_t)(lev * O_.niters), O_.niters));
  };
  dev_->ok(tsa_upload(c, init.data()));
  sweep_all(c);
  std::vector<uint64_t> fin(init.size());
  dev_->ok(tsa_download(c, 0, O_.nchains, fin.data()));
  uint64_t st[7], ch[2];
  dev_->counters(st, ch);
  const std::string desc = dev_->describe();
  printf("check: %d chains, %zu levels x %d sweeps, kernel %s (%s), mode %d, W=%d (64-bit words), slicing %d (moves %d): "
         "%llu proposals, %llu accepted, %llu/%llu slice moves accepted\n",
         O_.nchains, sched_.size(), O_.niters, kernel_label().c_str(), desc.c_str(), O_.mode, lay_.W, cfg_.slicing,
         cfg_.slice_moves, (unsigned long long)st[0], (unsigned long long)st[1], (unsigned long long)st[5],
         (unsigned long long)st[4]);
  int bad_tree = 0, bad_lab = 0, changed = 0, s_changed = 0;
  std::vector<uint64_t> lab((size_t)lay_.nint * lay_.W);
  for (int k = 0; k < O_.nchains; k++) {
    const uint64_t* r = &fin[(size_t)k * lay_.chain_words];
    const uint64_t* r0 = &init[(size_t)k * lay_.chain_words];
    if (!topology_labels(N_, lay_.W, children(r), lab.data())) {
      bad_tree++;
      continue;
    }
    bad_lab += !std::equal(lab.begin(), lab.end(), r);
    changed += !std::equal(r, r + lay_.s_off, r0);
    s_changed += !std::equal(r + lay_.s_off, r + lay_.s_off + lay_.W, r0 + lay_.s_off);
  }
  printf("  [1] invalid trees: %d, chains with label mismatch vs recomputation: %d (chains changed by SA: %d/%d, "
         "slice set changed: %d)\n",
         bad_tree, bad_lab, changed, O_.nchains, s_changed);
  Energies e(O_.nchains);
  dev_->ok(tsa_energy(c, e.lc.data(), e.sc.data(), e.ns.data()));
  double worst = 0;
  int sc_bad = 0;
  for (int k = 0; k < O_.nchains; k++) {
    const uint64_t* r = &fin[(size_t)k * lay_.chain_words];
    const HostEnergy H = host_energy(N_, lay_.W, model_, r, children(r), leaf_, slices(r));
    const double want = O_.mode == 0 ? H.tc : std::log2(O_.mode == 1 ? H.time : H.time2);
    worst = std::max(worst, std::fabs(want - (double)e.lc[k]));
    sc_bad += H.sc != e.sc[k] || H.ns != e.ns[k];
  }
  printf("  [2] GPU energy kernel vs host double: max |dlog2cost| = %.3g, sc/|S| mismatches %d\n", worst, sc_bad);
  int xdiff = -1;
  const bool is_lds = desc.compare(0, 3, "lds") == 0, is_wide = desc.compare(0, 4, "wide") == 0;
  if (O_.cross && cfg_.slice_moves == 0 && (is_lds || (is_wide && order_ == TSA_ORDER_PAR))) {
    tsa_config_t c2 = cfg_;
    c2.kernel = TSA_KERNEL_GLOBAL;
    Device other(lay_, leaf_, N_.largest_tensor(), c2, O_.nchains);
    other.ok(tsa_upload(other.get(), init.data()));
    for (size_t lev = 0; lev < sched_.size(); lev++)
      other.ok(tsa_sweeps(other.get(), order_, sched_[lev].beta, (uint32_t)(lev * O_.niters), O_.niters));
    std::vector<uint64_t> fin2(fin.size());
    other.ok(tsa_download(other.get(), 0, O_.nchains, fin2.data()));
    xdiff = 0;
    for (int k = 0; k < O_.nchains; k++)
      xdiff += !std::equal(fin.begin() + (size_t)k * lay_.chain_words, fin.begin() + (size_t)(k + 1) * lay_.chain_words,
                           fin2.begin() + (size_t)k * lay_.chain_words);
    printf("  [3] kernel %s vs global: chains differing: %d/%d\n", is_lds ? "lds" : "wide", xdiff, O_.nchains);
  }
  printf("  [4] CPU reference: not linked into this binary\n");
  const bool ok = bad_tree == 0 && bad_lab == 0 && sc_bad == 0 && worst < 1e-3 && xdiff <= 0;
  printf("CHECK %s\n", ok ? "PASSED" : "FAILED");
  return ok ? 0 : 3;
}

}  // namespace

int main(int argc, char** argv) {
  Options O;
  try {
    O = parse_options(argc, argv);
  } catch (const UsageError& e) {
    fprintf(stderr, "%s\n%s", e.what(), usage_text().c_str());
    return 1;
  }
  try {
    const Network N = read_network(O.instance);
    if (N.m < 3) throw InputError("need at least 3 tensors");
    if (2 * N.m - 1 > 65535) throw InputError("too many tensors (node ids are 16-bit)");
    Run R(N, O);
    return O.check ? R.check() : R.anneal();
  } catch (const InputError& e) {
    fprintf(stderr, "%s\n", e.what());
  } catch (const DeviceError& e) {
    fprintf(stderr, "%s\n", e.what());
  } catch (const std::bad_alloc&) {
    fprintf(stderr, "out of host memory\n");
  }
  return 1;
}
