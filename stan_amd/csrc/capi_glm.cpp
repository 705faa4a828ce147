// C-ABI for the GLM log density + gradient engine (declared in
// include/stanx.h).  Owns the device copies of X and y in the tiled layout,
// a private HIP stream, pinned staging buffers and the kernel choice.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <mutex>
#include <new>
#include <sstream>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "sx_internal.hpp"

namespace sx {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string& msg) { g_last_error = msg; }

}  // namespace sx

using sx::set_error;

namespace {

// compiled register capacities are the multiples of 4 up to 32
int smax_for(int64_t S) {
  int smax = 4;
  while (smax < S) smax += 4;
  return smax;
}

// lanes per row: fewest lanes whose register tile fits 32 slots
int default_lanes(int64_t K) {
  int L = 1;
  while (L < 64 && (K + L - 1) / L > 32) L <<= 1;
  return L;
}

int device_cus(int* cus) {
  int dev = 0;
  SX_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  SX_HIP(hipGetDeviceProperties(&prop, dev));
  *cus = prop.multiProcessorCount;
  return SX_OK;
}

// Size of a context's pinned output buffer at least: batches whose points and
// results each stay below it go through that buffer, so their first call pins
// nothing (pinning took 20 of the 73 us of a context's first 8-chain batch).
constexpr size_t kSmallBytes = size_t(64) << 10;

int clamp_blocks(const sx_glm* m, int blocks) {
  const int64_t max_blocks = std::max<int64_t>(1, (m->geom.T + 3) / 4);
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(blocks, max_blocks)));
}

int retile(sx_glm* m, const double* d_rowmajor, int L, int smax, int prefetch) {
  sx::tile_geom g = sx::make_geom(m->N, m->K, L, smax);
  g.prefetch = prefetch;
  const size_t need = static_cast<size_t>(g.T) * g.S * 64;
  const size_t have = static_cast<size_t>(m->geom.T) * m->geom.S * 64;
  if (need != have || (!m->d_X && need)) {
    if (m->d_X) (void)hipFree(m->d_X);
    m->d_X = nullptr;
    if (need) SX_HIP(hipMalloc(&m->d_X, need * sizeof(double)));
  }
  if (need) SX_HIP(sx::launch_tile_x_f64(d_rowmajor, m->d_X, m->N, m->K, g, m->stream));
  m->geom = g;
  return SX_OK;
}

}  // namespace

// forward declarations used by the autotuner
namespace {
int enqueue_pass(sx_glm* m, int propto, int jacobian, bool reduce = true);
}

namespace {

// The autotuner's decisions, one per device model and data shape.  The
// layout (lanes per row) and the block count set the order of the FP64
// sums, so the gradient's last bits depend on the choice; timing alone
// could choose differently in two contexts of the same data.  The first
// decision for a (device, family, N, K) is therefore kept for the process
// and reused by every later context, which makes two autotuned contexts of
// one data set bitwise equal.  With STANX_TUNING_CACHE naming a file, the
// decisions are also read from and appended to it, so that separate
// processes (e.g. seeded reruns) share them too.
struct tuned {
  int L, smax, pf, blocks;
};
std::mutex g_tune_mu;
std::map<std::string, tuned> g_tuned;
bool g_tune_file_read = false;

std::string tune_key(int device, int family, int64_t N, int64_t K) {
  hipDeviceProp_t prop;
  std::string arch = "dev";
  if (hipGetDeviceProperties(&prop, device) == hipSuccess)
    arch = std::string(prop.gcnArchName) + "/" + std::to_string(prop.multiProcessorCount);
  std::ostringstream k;
  k << arch << " " << family << " " << N << " " << K;
  return k.str();
}

// caller holds g_tune_mu
void read_tune_file() {
  if (g_tune_file_read) return;
  g_tune_file_read = true;
  const char* path = std::getenv("STANX_TUNING_CACHE");
  if (!path) return;
  std::ifstream f(path);
  std::string arch;
  int fam, L, smax, pf, blocks;
  long long N, K;
  while (f >> arch >> fam >> N >> K >> L >> smax >> pf >> blocks) {
    std::ostringstream k;
    k << arch << " " << fam << " " << N << " " << K;
    g_tuned.emplace(k.str(), tuned{L, smax, pf, blocks});
  }
}

void remember_tuning(const std::string& key, const tuned& t) {
  g_tuned.emplace(key, t);
  if (const char* path = std::getenv("STANX_TUNING_CACHE")) {
    std::ofstream f(path, std::ios::app);
    f << key << " " << t.L << " " << t.smax << " " << t.pf << " " << t.blocks << "\n";
  }
}

// Times candidate layouts / launch shapes on the device and keeps the
// fastest.  X is re-tiled from the row-major staging copy per layout.
int autotune(sx_glm* m, const double* d_rowmajor, int cus) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  read_tune_file();
  const std::string key = tune_key(m->device, m->family, m->N, m->K);
  const auto hit = g_tuned.find(key);
  if (hit != g_tuned.end()) {
    const tuned& t = hit->second;
    int rc = retile(m, d_rowmajor, t.L, t.smax, t.pf);
    if (rc) return rc;
    m->blocks = clamp_blocks(m, t.blocks);
    char line[160];
    std::snprintf(line, sizeof line,
                  "cached: L=%d smax=%d prefetch=%d blocks=%d (the first decision for %s)\n",
                  t.L, t.smax, t.pf, m->blocks, key.c_str());
    m->tuning_log = line;
    return SX_OK;
  }
  std::string log;
  std::vector<double> zeros(static_cast<size_t>(m->D), 0.0);
  SX_HIP(hipMemcpy(m->d_theta, zeros.data(), zeros.size() * sizeof(double),
                   hipMemcpyHostToDevice));
  struct cand { int L, smax, pf, blocks; double ms; };
  cand best{0, 0, 0, 0, 1e30};
  for (int L = 1; L <= 64; L <<= 1) {
    const int64_t S = (m->K + L - 1) / L;
    if (S > 32) continue;
    const double waste = static_cast<double>(S * L - m->K) / std::max<int64_t>(1, m->K);
    if (waste > 0.15 && L != default_lanes(m->K)) continue;
    const int smax = smax_for(S);
    for (int pf = 0; pf <= 1; ++pf) {
      int rc = retile(m, d_rowmajor, L, smax, pf);
      if (rc) return rc;
      for (int mult : {1, 2, 3, 4, 6, 8}) {
        m->blocks = clamp_blocks(m, mult * cus);
        if (mult > 1 && m->blocks < mult * cus) break;
        for (int w = 0; w < 2; ++w) {
          rc = enqueue_pass(m, 1, 1);
          if (rc) return rc;
        }
        SX_HIP(hipEventRecord(m->ev0, m->stream));
        const int reps = 5;
        for (int i = 0; i < reps; ++i) {
          rc = enqueue_pass(m, 1, 1);
          if (rc) return rc;
        }
        SX_HIP(hipEventRecord(m->ev1, m->stream));
        SX_HIP(hipEventSynchronize(m->ev1));
        float ms = 0.f;
        SX_HIP(hipEventElapsedTime(&ms, m->ev0, m->ev1));
        const double per = ms / reps;
        char line[160];
        std::snprintf(line, sizeof line, "L=%d S=%d smax=%d prefetch=%d blocks=%d: %.4f ms\n",
                      L, static_cast<int>(S), smax, pf, m->blocks, per);
        log += line;
        if (per < best.ms) best = cand{L, smax, pf, m->blocks, per};
      }
    }
  }
  int rc = retile(m, d_rowmajor, best.L, best.smax, best.pf);
  if (rc) return rc;
  m->blocks = best.blocks;
  remember_tuning(key, tuned{best.L, best.smax, best.pf, best.blocks});
  char line[160];
  std::snprintf(line, sizeof line, "chosen: L=%d smax=%d prefetch=%d blocks=%d (%.4f ms)\n",
                best.L, best.smax, best.pf, best.blocks, best.ms);
  log += line;
  m->tuning_log = log;
  return SX_OK;
}

// Hierarchical model: cut every group into chunks of at most `chunk` rows
// (a chunk never straddles a group) and upload the chunk tables.
int hier_chunks(sx_glm* m, const int64_t* off, int chunk) {
  std::vector<int> cg;
  std::vector<int64_t> cr0, gc0;
  gc0.reserve(static_cast<size_t>(m->J) + 1);
  for (int64_t j = 0; j < m->J; ++j) {
    gc0.push_back(static_cast<int64_t>(cg.size()));
    for (int64_t r = off[j]; r < off[j + 1]; r += chunk) {
      cg.push_back(static_cast<int>(j));
      cr0.push_back(r);
    }
  }
  gc0.push_back(static_cast<int64_t>(cg.size()));
  (void)hipFree(m->d_group_chunk0);
  (void)hipFree(m->d_by_rows);
  m->d_by_rows = nullptr;
  m->d_group_chunk0 = nullptr;
  m->n_chunks = static_cast<int64_t>(cg.size());
  m->hier_chunk = chunk;
  SX_HIP(hipMalloc(&m->d_group_chunk0, sizeof(int64_t) * gc0.size()));
  SX_HIP(hipMemcpy(m->d_group_chunk0, gc0.data(), sizeof(int64_t) * gc0.size(), hipMemcpyHostToDevice));
  if (!cg.empty()) {
    // most rows first, by a counting sort over the rows (1 .. chunk)
    std::vector<int64_t> at(static_cast<size_t>(chunk) + 1, 0);
    const auto rows = [&](size_t i) {  // a group's last chunk ends with the group
      return static_cast<int>(std::min<int64_t>(off[cg[i] + 1] - cr0[i], chunk));
    };
    for (size_t i = 0; i < cg.size(); ++i) ++at[chunk - rows(i)];
    int64_t sum = 0;
    for (int64_t& v : at) sum += std::exchange(v, sum);
    std::vector<sx::hier_chunk> t(cg.size());
    for (size_t i = 0; i < cg.size(); ++i)
      t[at[chunk - rows(i)]++] = {cr0[i], rows(i), cg[i], static_cast<int>(i), 0};
    SX_HIP(hipMalloc(&m->d_by_rows, sizeof(sx::hier_chunk) * t.size()));
    SX_HIP(hipMemcpy(m->d_by_rows, t.data(), sizeof(sx::hier_chunk) * t.size(),
                     hipMemcpyHostToDevice));
  }
  return SX_OK;
}

// Chunk size and FP32 product kernel of the hierarchical model, timed on
// the device at context creation: 128, 256, 512 or 1024 rows, and for an
// FP32 context with K <= 31 the FP32 MFMA products or the BF16 three-term
// split products, each timed as full evaluations at theta = 0 (the
// kernels' work does not depend on the values) -- one chain in FP64 for an
// FP64 context, a batch of 64 chains for an FP32 one.  Both choices set
// the order (or rounding) of sums, so the first decision per (device,
// precision, N, J, K, forced kernel) is kept for the process and in
// STANX_TUNING_CACHE (family field 200 + [FP32] + 10 x forced kernel, K
// field 64 J + K).
int hier_autotune(sx_glm* m, const int64_t* off, int kernel) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  read_tune_file();
  const bool fp32 = m->precision == SX_FP32;
  const std::string key =
      tune_key(m->device, 200 + (fp32 ? 1 : 0) + 10 * kernel, m->N, 64 * m->J + m->K);
  const auto hit = g_tuned.find(key);
  if (hit != g_tuned.end()) {
    m->hier_x6 = hit->second.smax;
    char line[160];
    std::snprintf(line, sizeof line, "hierarchical chunk cached: %d rows, %s products\n",
                  hit->second.L, m->hier_x6 ? "BF16 split" : "FP32");
    m->tuning_log += line;
    return hier_chunks(m, off, hit->second.L);
  }
  const int C = fp32 ? 64 : 1;
  const int64_t D = m->D;
  double *d_th = nullptr, *d_out = nullptr;
  if (hipMalloc(&d_th, sizeof(double) * C * D) != hipSuccess ||
      hipMalloc(&d_out, sizeof(double) * C * (D + 2)) != hipSuccess) {
    (void)hipFree(d_th);
    set_error("hierarchical autotune: out of device memory");
    return SX_ENOMEM;
  }
  int rc = hipMemsetAsync(d_th, 0, sizeof(double) * C * D, m->stream) == hipSuccess
               ? SX_OK : SX_EDEVICE;
  std::string log;
  int best_c = sx::kHierChunk, best_k = 0;
  double best_ms = 1e30;
  const bool can_x6 = fp32 && m->K <= 31;
  const int k_lo = kernel == 2 && can_x6 ? 1 : 0;
  const int k_hi = kernel == 1 || !can_x6 ? 0 : 1;
  for (int cand = 0; cand < 4 * (k_hi - k_lo + 1); ++cand) {
    const int chunk = 128 << (cand / (k_hi - k_lo + 1));
    const int kx6 = k_lo + cand % (k_hi - k_lo + 1);
    if (rc) break;
    m->hier_x6 = kx6;
    rc = hier_chunks(m, off, chunk);
    if (rc) break;
    sx::hier_workspace w;
    for (int i = 0; i < 2 && rc == SX_OK; ++i)
      rc = sx::hier_enqueue(m, w, d_th, C, d_out, 1, 1, fp32, m->stream);
    float ms = 0.f;
    const int reps = 5;
    if (rc == SX_OK && hipEventRecord(m->ev0, m->stream) != hipSuccess) rc = SX_EDEVICE;
    for (int i = 0; i < reps && rc == SX_OK; ++i)
      rc = sx::hier_enqueue(m, w, d_th, C, d_out, 1, 1, fp32, m->stream);
    if (rc == SX_OK && (hipEventRecord(m->ev1, m->stream) != hipSuccess ||
                        hipEventSynchronize(m->ev1) != hipSuccess ||
                        hipEventElapsedTime(&ms, m->ev0, m->ev1) != hipSuccess))
      rc = SX_EDEVICE;
    (void)hipStreamSynchronize(m->stream);
    sx::free_workspace(w);
    if (rc) break;
    const double per = ms / reps;
    char line[160];
    std::snprintf(line, sizeof line,
                  "hierarchical chunk=%d rows (%lld chunks)%s: %.4f ms (%d chain%s)\n", chunk,
                  static_cast<long long>(m->n_chunks), fp32 ? (kx6 ? ", BF16 split products" : ", FP32 products") : "",
                  per, C, C > 1 ? "s" : "");
    log += line;
    if (per < best_ms) {
      best_ms = per;
      best_c = chunk;
      best_k = kx6;
    }
  }
  m->hier_x6 = best_k;
  (void)hipFree(d_th);
  (void)hipFree(d_out);
  m->tuning_log += log;
  if (rc) return rc;
  remember_tuning(key, tuned{best_c, best_k, 0, 0});
  char line[160];
  std::snprintf(line, sizeof line, "hierarchical chunk chosen: %d rows, %s products (%.4f ms)\n",
                best_c, best_k ? "BF16 split" : "FP32", best_ms);
  m->tuning_log += line;
  return hier_chunks(m, off, best_c);
}

// Hierarchical model: the chunk tables (the caller's chunk size, else the
// autotuned one, else kHierChunk), an FP32 copy of X for batched evaluations (SX_FP32), and the
// single-chain partials.  The FP32 copy is sign-folded: row n holds
// (2 y_n - 1) x_n.
int hier_setup(sx_glm* m, const double* d_X, const double* X, const int32_t* y,
               const int64_t* off, bool do_tune, int chunk, int kernel) {
  if (m->precision == SX_FP32 && m->N > 0) {
    // 32 K + 64 zero floats past the last row: the FP32 pass stages whole
    // 32-row tiles (64-float loads per lane) past a chunk's end
    const size_t n = static_cast<size_t>(m->N * m->K);
    const size_t K = static_cast<size_t>(m->K);
    const size_t total = n + 32 * K + 64;
    std::vector<float> x32(total, 0.0f);
    for (size_t i = 0; i < n; ++i) {
      const float v = static_cast<float>(X[i]);
      x32[i] = y[i / K] ? v : -v;
    }
    if (n > 0) {
      SX_HIP(hipMalloc(&m->d_X32, total * sizeof(float)));
      SX_HIP(hipMemcpy(m->d_X32, x32.data(), total * sizeof(float), hipMemcpyHostToDevice));
    }
    if (K <= 31) {
      // the x6 pass's copy: per row and term t, columns 0 .. 8 NCH - 1 of
      // (x'_0 .. x'_{K-1}, s, 0 ...) as term t of the exact three-term
      // BF16 split by truncation (h = x with the low 16 bits cleared,
      // m = (x - h) likewise, l = x - h - m), 32 zero rows past the last
      const size_t W = 8 * static_cast<size_t>(sx::hier_x6_chunks(static_cast<int>(K)));
      const size_t N = static_cast<size_t>(m->N);
      std::vector<uint16_t> xs((N + 32) * 3 * W, 0);
      auto bits = [](float f) {
        uint32_t u;
        std::memcpy(&u, &f, 4);
        return u;
      };
      auto from_bits = [](uint32_t u) {
        float f;
        std::memcpy(&f, &u, 4);
        return f;
      };
      for (size_t r = 0; r < N; ++r) {
        uint16_t* row = xs.data() + r * 3 * W;
        for (size_t c = 0; c <= K; ++c) {
          const float v = c < K ? x32[r * K + c] : (y[r] ? 1.0f : -1.0f);
          const uint32_t h = bits(v) & 0xffff0000u;
          const float r1 = v - from_bits(h);
          const uint32_t mm = bits(r1) & 0xffff0000u;
          const uint32_t l = bits(r1 - from_bits(mm));
          row[c] = static_cast<uint16_t>(h >> 16);
          row[W + c] = static_cast<uint16_t>(mm >> 16);
          row[2 * W + c] = static_cast<uint16_t>(l >> 16);
        }
      }
      SX_HIP(hipMalloc(&m->d_XS, xs.size() * sizeof(uint16_t)));
      SX_HIP(hipMemcpy(m->d_XS, xs.data(), xs.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
    }
  }
  m->d_X = const_cast<double*>(d_X);  // the FP64 pass reads X row-major
  // FP32 products unless asked for (or timed) otherwise
  m->hier_x6 = kernel == 2 && m->precision == SX_FP32 && m->K <= 31 ? 1 : 0;
  const int rc = chunk > 0 ? hier_chunks(m, off, chunk)
                 : do_tune && m->N * m->K > 0 ? hier_autotune(m, off, kernel)
                                              : hier_chunks(m, off, sx::kHierChunk);
  if (rc) return rc;
  return sx::hier_prepare(m, m->hw, 1);
}

}  // namespace

extern "C" {

const char* sx_last_error(void) { return sx::g_last_error.c_str(); }

int sx_glm_create(sx_glm** out, int family, const double* X, const void* y, int64_t N,
                  int64_t K, const int64_t* group_offsets, int64_t J, int precision,
                  const sx_prior* prior, int device) {
  return sx_glm_create_ex(out, family, X, y, N, K, group_offsets, J, precision, prior, device,
                          nullptr);
}

int sx_glm_create_ex(sx_glm** out, int family, const double* X, const void* y, int64_t N,
                     int64_t K, const int64_t* group_offsets, int64_t J, int precision,
                     const sx_prior* prior, int device, const sx_tuning* tuning) {
  if (!out) {
    set_error("sx_glm_create: out is NULL");
    return SX_EINVAL;
  }
  *out = nullptr;
  if (family != SX_LOGIT && family != SX_NORMAL && family != SX_HIER_LOGIT) {
    set_error("sx_glm_create: unknown family");
    return SX_EINVAL;
  }
  const bool hier = family == SX_HIER_LOGIT;
  if ((!hier && precision != SX_FP64 && precision != SX_BF16X2) ||
      (hier && precision != SX_FP64 && precision != SX_FP32)) {
    set_error("sx_glm_create: precision not supported for this family");
    return SX_EINVAL;
  }
  if (hier) {
    if (K > 32) {
      set_error("sx_glm_create: the hierarchical model supports K <= 32");
      return SX_EINVAL;
    }
    if (J < 1 || !group_offsets) {
      set_error("sx_glm_create: the hierarchical model needs J >= 1 group offsets");
      return SX_EINVAL;
    }
    if (group_offsets[0] != 0 || group_offsets[J] != N) {
      set_error("sx_glm_create: group offsets must start at 0 and end at N");
      return SX_EINVAL;
    }
    for (int64_t j = 0; j < J; ++j)
      if (group_offsets[j + 1] < group_offsets[j]) {
        set_error("sx_glm_create: group offsets must be non-decreasing");
        return SX_EINVAL;
      }
  }
  if (precision == SX_BF16X2 && K > 512) {
    set_error("sx_glm_create: BF16 hi+lo batched evaluation supports K <= 512");
    return SX_EINVAL;
  }
  if (N < 0 || K < 0 || K > 1024 || (N > 0 && (!X || !y))) {
    set_error("sx_glm_create: invalid sizes or NULL data");
    return SX_EINVAL;
  }
  sx_tuning tune{0, 0, -1, 0, -1, 0, 0};
  if (tuning) tune = *tuning;
  if (tune.lanes_per_row < 0 || tune.lanes_per_row > 64 ||
      (tune.lanes_per_row & (tune.lanes_per_row - 1)) != 0 ||
      tune.slots_cap < 0 || tune.slots_cap > 32 || tune.slots_cap % 4 != 0 ||
      tune.prefetch < -1 || tune.prefetch > 1 || tune.blocks < 0 || tune.hier_chunk < 0 ||
      tune.hier_chunk > 4096 || tune.hier_chunk % 32 != 0 || tune.hier_kernel < 0 ||
      tune.hier_kernel > 2) {
    set_error("sx_glm_create: invalid tuning");
    return SX_EINVAL;
  }
  // data checks the reference's GLM functions perform (y in {0,1},
  // finite y and X) happen once here instead of per evaluation
  if (family == SX_LOGIT || hier) {
    const int32_t* yi = static_cast<const int32_t*>(y);
    for (int64_t n = 0; n < N; ++n)
      if (yi[n] != 0 && yi[n] != 1) {
        set_error(std::string(hier ? "bernoulli_logit" : "bernoulli_logit_glm") + ": y[" + std::to_string(n) + "] is " +
                  std::to_string(yi[n]) + ", but must be in {0, 1}");
        return SX_EINVAL;
      }
  } else {
    const double* yd = static_cast<const double*>(y);
    for (int64_t n = 0; n < N; ++n)
      if (!std::isfinite(yd[n])) {
        set_error("normal_id_glm: y[" + std::to_string(n) + "] is not finite");
        return SX_EINVAL;
      }
  }
  for (int64_t i = 0; i < N * K; ++i)
    if (!std::isfinite(X[i])) {
      set_error("GLM: X contains a non-finite value");
      return SX_EINVAL;
    }
  int ndev = 0;
  SX_HIP(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev) {
    set_error("sx_glm_create: no such device");
    return SX_EINVAL;
  }
  SX_HIP(hipSetDevice(device));
  int cus = 0;
  int rc = device_cus(&cus);
  if (rc) return rc;
  // the allocation-free entry point's scratch address on this device (its
  // failure only disables that entry point, which then reports it)
  (void)sx::noalloc_setup(device);
  sx_glm* m = new sx_glm();
  m->family = family;
  m->precision = precision;
  m->device = device;
  m->N = N;
  m->K = K;
  m->J = J;
  m->D = family == SX_LOGIT ? K + 1 : family == SX_NORMAL ? K + 2 : 2 * K + 2 + J * (K + 1);
  m->prior = prior ? *prior : sx_prior{5.0, 2.0, 2.0, 1.0};
  auto fail = [&](int code) {
    sx_glm_destroy(m);
    return code;
  };
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) {
    set_error("hipStreamCreate failed");
    delete m;
    return SX_EDEVICE;
  }
  if (family == SX_LOGIT || hier) {
    std::vector<int8_t> y8(static_cast<size_t>(std::max<int64_t>(N, 1)));
    const int32_t* yi = static_cast<const int32_t*>(y);
    for (int64_t n = 0; n < N; ++n) y8[n] = static_cast<int8_t>(yi[n]);
    if (hipMalloc(&m->d_y, y8.size()) != hipSuccess) return fail(SX_ENOMEM);
    if (hipMemcpy(m->d_y, y8.data(), y8.size(), hipMemcpyHostToDevice) != hipSuccess)
      return fail(SX_EDEVICE);
  } else {
    const size_t bytes = sizeof(double) * static_cast<size_t>(std::max<int64_t>(N, 1));
    if (hipMalloc(&m->d_y, bytes) != hipSuccess) return fail(SX_ENOMEM);
    if (N && hipMemcpy(m->d_y, y, sizeof(double) * N, hipMemcpyHostToDevice) != hipSuccess)
      return fail(SX_EDEVICE);
  }
  if (hipMalloc(&m->d_theta, sizeof(double) * (m->D + 1)) != hipSuccess) return fail(SX_ENOMEM);
  if (hipMalloc(&m->d_out, sizeof(double) * (m->D + 2)) != hipSuccess) return fail(SX_ENOMEM);
  if (hipHostMalloc(&m->h_theta, sizeof(double) * (m->D + 1)) != hipSuccess) return fail(SX_ENOMEM);
  // the kernels' stores reach it while they run, whatever the process's default
  if (hipHostMalloc(&m->h_out, std::max(sizeof(double) * (m->D + 2), kSmallBytes),
                    hipHostMallocCoherent) != hipSuccess)
    return fail(SX_ENOMEM);
  if (hipEventCreate(&m->ev0) != hipSuccess || hipEventCreate(&m->ev1) != hipSuccess)
    return fail(SX_EDEVICE);
  const int max_blocks = 8 * cus;
  const size_t E = static_cast<size_t>(K) + 3;
  if (hipMalloc(&m->d_partials, sizeof(double) * max_blocks * E) != hipSuccess)
    return fail(SX_ENOMEM);
  m->max_blocks = max_blocks;

  // row-major staging copy on the device, tiled into the kernel layout (the
  // hierarchical model keeps it, with 64 K zero doubles past the last row:
  // its FP64 pass loads whole 64-row blocks past a chunk's end)
  double* staging = nullptr;
  if (N * K > 0) {
    const size_t pad = hier ? static_cast<size_t>(64 * K) : 0;
    if (hipMalloc(&staging, (static_cast<size_t>(N * K) + pad) * sizeof(double)) != hipSuccess) {
      set_error("hipMalloc(staging X) failed");
      return fail(SX_ENOMEM);
    }
    if (hipMemcpy(staging, X, static_cast<size_t>(N * K) * sizeof(double),
                  hipMemcpyHostToDevice) != hipSuccess ||
        (pad > 0 && hipMemset(staging + N * K, 0, pad * sizeof(double)) != hipSuccess)) {
      (void)hipFree(staging);
      set_error("X upload failed");
      return fail(SX_EDEVICE);
    }
  }
  const bool do_tune =
      tune.autotune == 1 || (tune.autotune == -1 && tuning == nullptr && N * K >= (1 << 22));
  if (hier) {
    rc = hier_setup(m, staging, X, static_cast<const int32_t*>(y), group_offsets, do_tune,
                    tune.hier_chunk, tune.hier_kernel);
    if (rc == SX_OK && hipStreamSynchronize(m->stream) != hipSuccess) rc = SX_EDEVICE;
    if (rc) {
      m->d_X = nullptr;
      if (staging) (void)hipFree(staging);
      return fail(rc);
    }
    *out = m;
    return SX_OK;
  }
  if (do_tune && N * K > 0) {
    rc = autotune(m, staging, cus);
  } else {
    const int L = tune.lanes_per_row > 0 ? tune.lanes_per_row : default_lanes(K);
    const int64_t S = (K + L - 1) / L;
    const int smax = tune.slots_cap > 0 ? tune.slots_cap : smax_for(S);
    if (S > smax) {
      set_error("sx_glm_create: K does not fit lanes_per_row x slots_cap");
      rc = SX_EINVAL;
    } else {
      rc = retile(m, staging, L, smax, tune.prefetch == 1 ? 1 : 0);
      m->blocks = clamp_blocks(m, tune.blocks > 0 ? std::min(tune.blocks, max_blocks)
                                                  : 2 * cus);
    }
  }
  if (rc == SX_OK && precision == SX_BF16X2) {
    m->Np = (N + 31) / 32 * 32;
    // a multiple of 32 up to 256; above, of 64 (the adjoint's column
    // blocks of 128, a last one of 64)
    m->Kp = K <= 256 ? std::max<int64_t>(32, (K + 31) / 32 * 32) : (K + 63) / 64 * 64;
    const size_t elems = static_cast<size_t>(m->Np) * m->Kp;
    if (hipMalloc(&m->d_Xh, elems * 2) != hipSuccess || hipMalloc(&m->d_Xl, elems * 2) != hipSuccess ||
        hipMalloc(&m->d_yf, sizeof(float) * m->Np) != hipSuccess) {
      set_error("hipMalloc(BF16 X) failed");
      rc = SX_ENOMEM;
    } else if (sx::launch_split_x(staging, m->d_Xh, m->d_Xl, N, K, m->Np, m->Kp, m->stream) !=
                   hipSuccess ||
               sx::launch_prep_y(m->d_y, m->d_yf, family, N, m->Np, m->stream) != hipSuccess) {
      set_error("BF16 split of X failed");
      rc = SX_EDEVICE;
    } else if (do_tune && N * K > 0) {
      rc = sx::mx_autotune(m);
    }
  }
  if (rc == SX_OK && hipStreamSynchronize(m->stream) != hipSuccess) rc = SX_EDEVICE;
  if (staging) (void)hipFree(staging);
  if (rc) return fail(rc);
  *out = m;
  return SX_OK;
}

const char* sx_glm_tuning_log(const sx_glm* m) { return m ? m->tuning_log.c_str() : ""; }

void sx_glm_destroy(sx_glm* m) {
  if (!m) return;
  (void)hipSetDevice(m->device);
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  (void)hipFree(m->d_X);
  (void)hipFree(m->d_y);
  (void)hipFree(m->d_theta);
  (void)hipFree(m->d_partials);
  (void)hipFree(m->d_out);
  (void)hipFree(m->d_Xh);
  (void)hipFree(m->d_Xl);
  (void)hipFree(m->d_yf);
  sx::free_workspace(m->mx);
  (void)hipFree(m->d_btheta);
  (void)hipFree(m->d_bout);
  (void)hipFree(m->d_bpart);
  (void)hipFree(m->d_X32);
  (void)hipFree(m->d_XS);
  (void)hipFree(m->d_group_chunk0);
  (void)hipFree(m->d_by_rows);
  sx::free_workspace(m->hw);
  if (m->h_theta) (void)hipHostFree(m->h_theta);
  if (m->h_out) (void)hipHostFree(m->h_out);
  if (m->h_batch) (void)hipHostFree(m->h_batch);
  if (m->ev0) (void)hipEventDestroy(m->ev0);
  if (m->ev1) (void)hipEventDestroy(m->ev1);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
}

int sx_glm_num_params(const sx_glm* m, int64_t* D) {
  if (!m || !D) {
    set_error("sx_glm_num_params: NULL argument");
    return SX_EINVAL;
  }
  *D = m->D;
  return SX_OK;
}

int sx_glm_family(const sx_glm* m) { return m ? m->family : -1; }

int sx_glm_dims(const sx_glm* m, int64_t* N, int64_t* K, int64_t* J) {
  if (!m) {
    set_error("sx_glm_dims: NULL model");
    return SX_EINVAL;
  }
  if (N) *N = m->N;
  if (K) *K = m->K;
  if (J) *J = m->J;
  return SX_OK;
}

}  // extern "C"

namespace {

int enqueue_pass(sx_glm* m, int propto, int jacobian, bool reduce) {
  if (m->family == SX_HIER_LOGIT)
    return sx::hier_enqueue(m, m->hw, m->d_theta, 1, m->d_out, propto, jacobian, false, m->stream);
  return sx::plain_enqueue(m, m->d_theta, m->d_out, m->d_partials, propto, jacobian, m->stream,
                           reduce);
}

// A word of the pinned output that no kernel has stored yet: a NaN with a
// payload that arithmetic on finite inputs does not produce.
constexpr uint64_t kUnset = 0x7ff4a5a55a5a0001ull;

void unset_words(double* w, size_t n) {
  for (size_t i = 0; i < n; ++i) std::memcpy(w + i, &kUnset, sizeof kUnset);
}

// Waits until the kernels on m's stream have stored n output words (each
// one aligned 8-byte store, so a word that is no longer kUnset is whole) and
// copies them to dst (unless NULL) as they arrive.
// Every word that is read must be among them: a word says nothing about
// another one, also not of an earlier launch, whose stores only the stream's
// completion publishes to the host.
// Watching the words returns a few microseconds before the stream's
// completion signal would (4 of 20 us for a small evaluation); 5 ms after
// `start` the stream is waited for instead, which also reports a failed
// launch.
int take_words(sx_glm* m, const double* w, size_t n, double* dst,
               std::chrono::steady_clock::time_point start) {
  bool synced = false;
  unsigned spins = 0;
  for (size_t i = 0; i < n;) {
    constexpr size_t kBlock = 64;
    uint64_t v[kBlock];  // what is copied is what was seen to be stored
    const size_t count = std::min(n - i, kBlock);
    bool any = false;
    for (size_t k = 0; k < count; ++k) {
      v[k] = __atomic_load_n(reinterpret_cast<const uint64_t*>(w + i + k), __ATOMIC_ACQUIRE);
      any |= v[k] == kUnset;
    }
    if (!any) {
      if (dst) std::memcpy(dst + i, v, count * sizeof(double));
      i += count;
    } else if (synced) {
      set_error("log_prob: the device stored no result");
      return SX_EDEVICE;
    } else if (++spins % 256 == 0 &&
               std::chrono::steady_clock::now() - start > std::chrono::milliseconds(5)) {
      SX_HIP(hipStreamSynchronize(m->stream));
      synced = true;
    } else {
      __builtin_ia32_pause();
    }
  }
  return SX_OK;
}

// A call that returns with an error leaves nothing queued: its copies read
// the caller's points, or buffers that the next call fills while it runs.
struct drain_on_error {
  sx_glm* m;
  bool done = false;
  ~drain_on_error() {
    if (!done) (void)hipStreamSynchronize(m->stream);
  }
};

const char* domain_message(int family) {
  return family == SX_LOGIT ? "bernoulli_logit_glm_lpmf: linear predictor or log density is not finite"
         : family == SX_NORMAL
             ? "normal_id_glm_lpdf: scale, linear predictor or log density is not finite"
             : "bernoulli_logit_lpmf: linear predictor or log density is not finite";
}

// index of the first non-finite value, or -1 (blocks are checked without an
// early exit, which the compiler vectorises)
int64_t first_non_finite(const double* x, int64_t n) {
  constexpr int64_t kBlock = 256;
  for (int64_t b = 0; b < n; b += kBlock) {
    const int64_t e = std::min(n, b + kBlock);
    int bad = 0;
    for (int64_t i = b; i < e; ++i) bad |= !(std::fabs(x[i]) <= 1.7976931348623157e308);
    if (bad)
      for (int64_t i = b; i < e; ++i)
        if (!std::isfinite(x[i])) return i;
  }
  return -1;
}

int eval(sx_glm* m, const double* theta, int propto, int jacobian, double* lp,
         double* grad) {
  if (!m || !theta || !lp) {
    set_error("NULL argument");
    return SX_EINVAL;
  }
  SX_HIP(hipSetDevice(m->device));
  const size_t D = static_cast<size_t>(m->D);
  if (const int64_t bad = first_non_finite(theta, m->D); bad >= 0) {
    set_error("log_prob: parameter " + std::to_string(bad) + " is not finite");
    return SX_EDOMAIN;
  }
  std::memcpy(m->h_theta, theta, D * sizeof(double));
  drain_on_error queued{m};
  int rc;
  if (m->family == SX_HIER_LOGIT) {
    // the words are reset while theta is on its way
    SX_HIP(hipMemcpyAsync(m->d_theta, m->h_theta, D * sizeof(double), hipMemcpyHostToDevice,
                          m->stream));
    unset_words(m->h_out, D + 2);
    rc = sx::hier_enqueue(m, m->hw, m->d_theta, 1, m->h_out, propto, jacobian, false, m->stream,
                          true);
  } else {
    unset_words(m->h_out, D + 2);
    rc = sx::plain_eval(m, propto, jacobian);
  }
  if (rc) return rc;
  // the words in the order in which they are stored: the hierarchical
  // model's z gradients come a launch before the others
  const auto start = std::chrono::steady_clock::now();
  const size_t head = m->family == SX_HIER_LOGIT ? 2 * static_cast<size_t>(m->K) + 3 : D + 1;
  rc = take_words(m, m->h_out + head, D + 1 - head, grad ? grad + head - 1 : nullptr, start);
  if (rc == SX_OK)
    rc = take_words(m, m->h_out + 1, head - 1, grad, start);
  if (rc == SX_OK) rc = take_words(m, m->h_out, 1, lp, start);
  double status = 0.0;
  if (rc == SX_OK) rc = take_words(m, m->h_out + D + 1, 1, &status, start);
  if (rc) return rc;
  queued.done = true;
  if (status != 0.0) {
    set_error(domain_message(m->family));
    return SX_EDOMAIN;
  }
  return SX_OK;
}

}  // namespace

namespace sx {

// Batched MFMA evaluation of C chains: theta (device, C x D) -> out
// (device, C x (D + 2)).  Row splits depend on N only, so each chain's
// result is independent of the other chains in the batch.
void free_workspace(mx_workspace& w) {
  (void)hipFree(w.Bh);
  (void)hipFree(w.Bl);
  (void)hipFree(w.Bm);
  (void)hipFree(w.Rh);
  (void)hipFree(w.Rl);
  (void)hipFree(w.alpha);
  (void)hipFree(w.gpart);
  (void)hipFree(w.spart);
  w = mx_workspace();
}

void free_workspace(hier_workspace& w) {
  (void)hipFree(w.cpart);
  (void)hipFree(w.gpart);
  (void)hipFree(w.wsplit);
  w = hier_workspace();
}

// Arguments of the FP64 pass of a logistic or normal context, one chain.
static pass_args plain_args(const sx_glm* m, const double* theta, double* out, double* partials,
                            int propto, int jacobian) {
  pass_args a;
  a.X = m->d_X;
  a.y = m->d_y;
  a.theta = theta;
  a.partials = partials;
  a.out = out;
  a.N = m->N;
  a.T = m->geom.T;
  a.K = static_cast<int>(m->K);
  a.L = m->geom.L;
  a.lgL = m->geom.lgL;
  a.S = m->geom.S;
  a.D = static_cast<int>(m->D);
  a.E = static_cast<int>(m->K) + 3;
  a.propto = propto;
  a.jacobian = jacobian;
  a.alpha_sd = m->prior.alpha_sd;
  a.beta_sd = m->prior.beta_sd;
  a.sigma_sd = m->prior.sigma_sd;
  a.sigma_mu = m->prior.sigma_mu;
  const double half_log_2pi = 0.91893853320467274178032973640562;
  a.alpha_const = a.alpha_sd > 0 ? -std::log(a.alpha_sd) - half_log_2pi : 0.0;
  a.beta_const = a.beta_sd > 0 ? -std::log(a.beta_sd) - half_log_2pi : 0.0;
  a.sigma_const = a.sigma_sd > 0 ? -std::log(a.sigma_sd) - half_log_2pi : 0.0;
  return a;
}

// The FP64 pass of a logistic or normal context: theta (device, chains x D)
// -> out (device, chains x (D + 2)), per-block partials in `partials`
// (chains x blocks x (K + 3) doubles), on `stream`.
int plain_enqueue(sx_glm* m, const double* d_theta, double* d_out, double* partials, int propto,
                  int jacobian, hipStream_t stream, bool reduce, int chains) {
  pass_args a = plain_args(m, d_theta, d_out, partials, propto, jacobian);
  a.chains = chains;
  a.theta_stride = m->D;
  a.out_stride = m->D + 2;
  SX_HIP(launch_pass_f64(m->family, m->geom, a, m->blocks, m->threads, stream, reduce));
  return SX_OK;
}

// The same evaluation from h_theta into h_out (pinned, D + 2), whose words
// the kernels store straight to host memory.
int plain_eval(sx_glm* m, int propto, int jacobian) {
  const pass_args a =
      plain_args(m, m->d_theta, m->h_out, m->d_partials, propto, jacobian);
  SX_HIP(launch_eval_f64(m->family, m->geom, a, m->h_theta, m->blocks, m->threads, m->stream));
  return SX_OK;
}

// chains padded to the chain tile of the MFMA kernel (32x32 tiles, waves
// of 32 chains): 64 for batches of at most 64 chains (two waves per
// workgroup), else a multiple of 128 (four waves)
int mx_chain_pad(const sx_glm* m, int C) {
  (void)m;
  if (C <= 64) return 64;
  return (C + 127) / 128 * 128;
}

// row splits for a target of tps tiles each: a multiple of 8, at most 512
static int mx_splits(const sx_glm* m, int64_t tps) {
  const int64_t n_tiles = m->Np / 32;
  if (tps <= 0) tps = 8;
  return static_cast<int>(
      std::min<int64_t>(512, std::max<int64_t>(8, ((n_tiles + tps - 1) / tps + 7) / 8 * 8)));
}

int mx_prepare(sx_glm* m, mx_workspace& w, int C) {
  if (!m->d_Xh) {
    set_error("batched BF16 evaluation needs a context created with SX_BF16X2");
    return SX_EINVAL;
  }
  const int Cp = mx_chain_pad(m, C);
  const int splits = mx_splits(m, m->mx_tps);
  if (w.cap >= Cp && w.splits == splits) return SX_OK;
  free_workspace(w);
  const size_t ck = static_cast<size_t>(Cp) * m->Kp;
  SX_HIP(hipMalloc(&w.Bh, ck * 2));
  SX_HIP(hipMalloc(&w.Bl, ck * 2));
  SX_HIP(hipMalloc(&w.Bm, ck * 2));
  SX_HIP(hipMalloc(&w.alpha, sizeof(float) * Cp));
  SX_HIP(hipMalloc(&w.gpart, sizeof(float) * ck * splits));
  SX_HIP(hipMalloc(&w.spart, sizeof(double) * 3 * static_cast<size_t>(Cp) * splits));
  if (m->Kp > 256) {  // residuals between the forward and the adjoint launch
    const size_t nr = static_cast<size_t>(m->Np) * Cp;
    SX_HIP(hipMalloc(&w.Rh, nr * 2));
    SX_HIP(hipMalloc(&w.Rl, nr * 2));
  }
  w.cap = Cp;
  w.Cp = Cp;
  w.splits = splits;
  return SX_OK;
}

int mx_enqueue(sx_glm* m, mx_workspace& w, const double* d_theta, int C, double* d_out,
               int propto, int jacobian, hipStream_t stream) {
  int rc = mx_prepare(m, w, C);
  if (rc) return rc;
  mx_args a{};
  a.Xh = m->d_Xh;
  a.Xl = m->d_Xl;
  a.y = m->d_y;
  a.yf = m->d_yf;
  a.Bh = w.Bh;
  a.Bl = w.Bl;
  a.Bm = w.Bm;
  a.alpha = w.alpha;
  a.gpart = w.gpart;
  a.spart = w.spart;
  a.Rh = w.Rh;
  a.Rl = w.Rl;
  a.N = m->N;
  a.n_tiles = m->Np / 32;
  a.Kp = static_cast<int>(m->Kp);
  a.Cp = mx_chain_pad(m, C);
  a.splits = w.splits;
  a.tiles_per_split = (a.n_tiles + a.splits - 1) / a.splits;
  a.variant = m->mx_variant;
  pass_args pa{};
  pa.theta = d_theta;
  pa.out = d_out;
  pa.N = m->N;
  pa.K = static_cast<int>(m->K);
  pa.D = static_cast<int>(m->D);
  pa.E = static_cast<int>(m->K) + 3;
  pa.propto = propto;
  pa.jacobian = jacobian;
  pa.chains = C;
  pa.theta_stride = m->D;
  pa.out_stride = m->D + 2;
  pa.alpha_sd = m->prior.alpha_sd;
  pa.beta_sd = m->prior.beta_sd;
  pa.sigma_sd = m->prior.sigma_sd;
  pa.sigma_mu = m->prior.sigma_mu;
  const double h = 0.91893853320467274178032973640562;
  pa.alpha_const = pa.alpha_sd > 0 ? -std::log(pa.alpha_sd) - h : 0.0;
  pa.beta_const = pa.beta_sd > 0 ? -std::log(pa.beta_sd) - h : 0.0;
  pa.sigma_const = pa.sigma_sd > 0 ? -std::log(pa.sigma_sd) - h : 0.0;
  SX_HIP(launch_mfma_pass(m->family, d_theta, m->D, C, a, pa, stream));
  return SX_OK;
}

// Row splits to time, as target tiles per split: 4 to 128 tiles, and those
// that give half, one and two splits per CU, so that the workgroups of one or
// two chain blocks fill whole rounds of the device (N = 2e5, K = 256: 200
// splits make 400 workgroups for 256 chains, 1.6 rounds of 256 CUs; 256
// splits make two).  Each split count once.
static std::vector<int> mx_split_targets(const sx_glm* m, int cus) {
  const int64_t n_tiles = m->Np / 32, per = std::max(1, cus);
  std::vector<int> targets, seen;
  for (int64_t t : {int64_t(4), int64_t(8), int64_t(16), int64_t(32), int64_t(64), int64_t(128),
                    (2 * n_tiles + per - 1) / per, (n_tiles + per - 1) / per,
                    (n_tiles + 2 * per - 1) / (2 * per)}) {
    t = std::max<int64_t>(1, t);
    const int sp = mx_splits(m, t);
    if (std::find(seen.begin(), seen.end(), sp) != seen.end()) continue;
    seen.push_back(sp);
    targets.push_back(static_cast<int>(t));
  }
  return targets;
}

// Launch shape of the batched MFMA pass, timed on the device at context
// creation: the kernel variant (one wave per 32-chain block; a pair of
// waves split by k where Kp / 32 is even and at most 8; or, for Kp <= 128,
// one wave per block without operand prefetch at two waves per SIMD, the
// same products as the first) and the row split
// (target tiles of 32 rows per split; at most 512 splits, so large N reach
// fewer splits, and fewer gradient partials to sum, only with the larger
// targets), each timed as full
// evaluations of 128 chains at theta = 0 (the kernels' work does not depend
// on the values).  The split sets the order of the FP64 sums, so, as for
// the FP64 pass, the first decision per (device, family, N, K) is kept for
// the process (and in STANX_TUNING_CACHE, as family + 100).  The choice
// does not depend on the batch size, so a chain's result stays independent
// of the other chains in its batch.
int mx_autotune(sx_glm* m) {
  std::lock_guard<std::mutex> lock(g_tune_mu);
  read_tune_file();
  const std::string key = tune_key(m->device, 100 + m->family, m->N, m->K);
  const auto hit = g_tuned.find(key);
  if (hit != g_tuned.end()) {
    m->mx_variant = hit->second.L;
    m->mx_tps = hit->second.smax;
    char line[160];
    std::snprintf(line, sizeof line, "MFMA pass cached: variant=%d tiles/split=%d\n",
                  m->mx_variant, m->mx_tps);
    m->tuning_log += line;
    return SX_OK;
  }
  const int C = 128;
  const int64_t D = m->D;
  double *d_th = nullptr, *d_out = nullptr;
  if (hipMalloc(&d_th, sizeof(double) * C * D) != hipSuccess ||
      hipMalloc(&d_out, sizeof(double) * C * (D + 2)) != hipSuccess) {
    (void)hipFree(d_th);
    set_error("MFMA autotune: out of device memory");
    return SX_ENOMEM;
  }
  mx_workspace w;
  std::string log;
  int rc = hipMemsetAsync(d_th, 0, sizeof(double) * C * D, m->stream) == hipSuccess
               ? SX_OK : SX_EDEVICE;
  const int kq = static_cast<int>(m->Kp / 32);
  int best_v = 0, best_t = 8;
  double best_ms = 1e30;
  int cus = 0;
  if (rc == SX_OK) rc = device_cus(&cus);
  const std::vector<int> targets = mx_split_targets(m, cus);
  for (int v = 0; v <= 2 && rc == SX_OK; ++v) {
    if (v == 1 && (m->Kp > 256 || kq % 2 != 0)) continue;
    if (v == 2 && kq > 4) continue;
    for (int tps : targets) {
      m->mx_variant = v;
      m->mx_tps = tps;
      for (int i = 0; i < 2 && rc == SX_OK; ++i)
        rc = mx_enqueue(m, w, d_th, C, d_out, 1, 1, m->stream);
      if (rc) break;
      if (hipEventRecord(m->ev0, m->stream) != hipSuccess) { rc = SX_EDEVICE; break; }
      const int reps = 3;
      for (int i = 0; i < reps && rc == SX_OK; ++i)
        rc = mx_enqueue(m, w, d_th, C, d_out, 1, 1, m->stream);
      if (rc) break;
      float ms = 0.f;
      if (hipEventRecord(m->ev1, m->stream) != hipSuccess ||
          hipEventSynchronize(m->ev1) != hipSuccess ||
          hipEventElapsedTime(&ms, m->ev0, m->ev1) != hipSuccess) {
        rc = SX_EDEVICE;
        break;
      }
      const double per = ms / reps;
      char line[160];
      std::snprintf(line, sizeof line, "MFMA pass variant=%d tiles/split=%d: %.4f ms (128 chains)\n",
                    v, tps, per);
      log += line;
      if (per < best_ms) {
        best_ms = per;
        best_v = v;
        best_t = tps;
      }
    }
  }
  (void)hipStreamSynchronize(m->stream);
  free_workspace(w);
  (void)hipFree(d_th);
  (void)hipFree(d_out);
  m->mx_variant = best_v;
  m->mx_tps = best_t;
  if (rc) return rc;
  remember_tuning(key, tuned{best_v, best_t, 0, 0});
  char line[160];
  std::snprintf(line, sizeof line, "MFMA pass chosen: variant=%d tiles/split=%d (%.4f ms)\n",
                best_v, best_t, best_ms);
  log += line;
  m->tuning_log += log;
  return SX_OK;
}

// Hierarchical model, C chains: theta (device, C x D) -> out (device,
// C x (D + 2)); FP64 X, or FP32 X with chains on lanes.
int hier_prepare(sx_glm* m, hier_workspace& w, int C) {
  if (w.cap >= C) return SX_OK;
  free_workspace(w);
  const size_t E = static_cast<size_t>(m->K) + 3, G = 2 * static_cast<size_t>(m->K) + 5;
  SX_HIP(hipMalloc(&w.cpart, sizeof(double) * E * std::max<int64_t>(1, m->n_chunks) * C));
  SX_HIP(hipMalloc(&w.gpart, sizeof(double) * G * m->J * C));
  if (m->precision == SX_FP32 && m->K <= 31) {
    // the coefficient kernel writes columns 0 .. K; the rest stay zero
    SX_HIP(hipMalloc(&w.wsplit, sizeof(uint16_t) * 96 * m->J * C));
    SX_HIP(hipMemset(w.wsplit, 0, sizeof(uint16_t) * 96 * m->J * C));
  }
  w.cap = C;
  return SX_OK;
}

int hier_enqueue(sx_glm* m, hier_workspace& w, const double* d_theta, int C, double* d_out,
                 int propto, int jacobian, bool fp32, hipStream_t stream, bool host_out) {
  if (fp32 && !m->d_X32 && m->N * m->K > 0) {
    set_error("FP32 evaluation needs a context created with SX_FP32");
    return SX_EINVAL;
  }
  int rc = hier_prepare(m, w, C);
  if (rc) return rc;
  hier_args a{};
  a.X = m->d_X;
  a.X32 = m->d_X32;
  a.XS = m->d_XS;
  a.y = static_cast<const int8_t*>(m->d_y);
  a.theta = d_theta;
  a.out = d_out;
  a.cpart = w.cpart;
  a.gpart = w.gpart;
  a.wsplit = w.wsplit;
  a.group_chunk0 = m->d_group_chunk0;
  a.by_rows = m->d_by_rows;
  a.simds = m->max_blocks / 2;
  a.n_chunks = m->n_chunks;
  a.theta_stride = m->D;
  a.out_stride = m->D + 2;
  a.J = static_cast<int>(m->J);
  a.K = static_cast<int>(m->K);
  a.D = static_cast<int>(m->D);
  a.E = static_cast<int>(m->K) + 3;
  a.G = 2 * static_cast<int>(m->K) + 5;
  a.chains = C;
  a.propto = propto;
  a.jacobian = jacobian;
  a.x6 = m->hier_x6;
  a.alpha_sd = m->prior.alpha_sd;
  a.beta_sd = m->prior.beta_sd;
  a.tau_sd = m->prior.tau_sd;
  const double h = 0.91893853320467274178032973640562;
  a.alpha_const = a.alpha_sd > 0 ? -std::log(a.alpha_sd) - h : 0.0;
  a.beta_const = a.beta_sd > 0 ? -std::log(a.beta_sd) - h : 0.0;
  a.tau_const = a.tau_sd > 0 ? -std::log(a.tau_sd) - h : 0.0;
  SX_HIP(launch_hier(a, fp32, stream, host_out));
  return SX_OK;
}

}  // namespace sx

namespace {

int ensure_batch_staging(sx_glm* m, int64_t C) {
  if (m->bcap >= C) return SX_OK;
  (void)hipFree(m->d_btheta);
  (void)hipFree(m->d_bout);
  m->d_btheta = nullptr;
  m->d_bout = nullptr;
  m->bcap = 0;
  SX_HIP(hipMalloc(&m->d_btheta, sizeof(double) * C * m->D));
  SX_HIP(hipMalloc(&m->d_bout, sizeof(double) * C * (m->D + 2)));
  m->bcap = C;
  return SX_OK;
}

// largest batch the pinned buffer holds, in bytes
constexpr size_t kPinnedBytes = size_t(64) << 20;

// Pinned buffer of the batch calls, kept by the context.  One for both ways:
// a batch's results are copied into it only after its points have left it
// (stream order), and pinning costs about 0.1 ms per MB at the first call.
int ensure_batch_pinned(sx_glm* m, int64_t C) {
  if (m->hbcap >= C) return SX_OK;
  if (m->h_batch) (void)hipHostFree(m->h_batch);
  m->h_batch = nullptr;
  m->hbcap = 0;
  SX_HIP(hipHostMalloc(&m->h_batch, sizeof(double) * C * (m->D + 2)));
  m->hbcap = C;
  return SX_OK;
}

// fn(0) .. fn(n - 1) on up to four threads when `bytes` of copying are worth
// them (a thread starts in about 15 us, a core copies about 10 KB/us)
template <class F>
void spread_rows(int64_t n, size_t bytes, F fn) {
  const int64_t nt = std::min<int64_t>({n, 4, static_cast<int64_t>(bytes >> 20)});
  std::vector<std::thread> th;
  int64_t done = 0;  // rows that threads have taken
  try {
    for (int64_t i = 0; i + 1 < nt; ++i) {
      const int64_t a = n * i / nt, b = n * (i + 1) / nt;
      th.emplace_back([=] {
        for (int64_t r = a; r < b; ++r) fn(r);
      });
      done = b;
    }
  } catch (...) {  // no more threads: this one takes the rest
  }
  for (int64_t r = done; r < n; ++r) fn(r);
  for (auto& t : th) t.join();
}

// Runs a batched evaluation of C chains in slabs of at most `slab`: points to
// the device, enqueue(n) for the kernels (d_btheta -> d_bout), results back
// to lp and grad.  checked: a chain at a non-finite theta is a domain error
// whose gradient is left as it was.  A chain with a domain error gets lp =
// -inf and the call reports SX_EDOMAIN.
//
// The host copies bound a large batch (64 x 21,042 parameters, 10.8 MB each
// way: 1670 us per call through the runtime's staging of pageable memory,
// 1060 through a pinned buffer filled and emptied by four threads, of which
// the kernels 88).  Batches below kSmallBytes go through the context's pinned
// output buffer (15 KB: 163 -> 155 us).  Between kSmallBytes and kLargeBytes a single thread reads what a
// copy engine has just written more slowly than the runtime's staging
// delivers it (528 KB: 302 us pageable, 307 pinned).
constexpr size_t kLargeBytes = size_t(1) << 20;

template <class F>
int batch_call(sx_glm* m, const double* theta, int64_t C, int64_t slab, bool checked,
               const char* message, double* lp, double* grad, F enqueue) {
  SX_HIP(hipSetDevice(m->device));
  const int64_t D = m->D;
  const size_t row = sizeof(double) * static_cast<size_t>(D);
  slab = std::max<int64_t>(
      1, std::min<int64_t>({C, slab, static_cast<int64_t>(kPinnedBytes / (row + 16))}));
  const size_t most = slab * (row + 16);
  int rc = ensure_batch_staging(m, slab);
  if (rc) return rc;
  double* pinned = most < kSmallBytes ? m->h_out : nullptr;
  if (most >= kLargeBytes) {
    if (ensure_batch_pinned(m, slab) == SX_OK)
      pinned = m->h_batch;
    else  // refused: pageable
      (void)hipGetLastError();
  }
  std::vector<double> pageable;
  int worst = SX_OK;
  drain_on_error queued{m};
  for (int64_t b = 0; b < C; b += slab) {
    const int64_t n = std::min(slab, C - b);
    const double* th = theta + b * D;
    const double* src = th;
    if (pinned) {
      spread_rows(n, n * row,
                  [=](int64_t c) { std::memcpy(pinned + c * D, th + c * D, row); });
      src = pinned;
    }
    SX_HIP(hipMemcpyAsync(m->d_btheta, src, n * row, hipMemcpyHostToDevice, m->stream));
    rc = enqueue(static_cast<int>(n));
    if (rc) return rc;
    if (!pinned && pageable.empty()) {  // its pages while the kernels run
      try {
        pageable.resize(most / sizeof(double));
      } catch (const std::bad_alloc&) {
        set_error("batched evaluation: out of host memory");
        return SX_ENOMEM;
      }
    }
    double* const out = pinned ? pinned : pageable.data();
    SX_HIP(hipMemcpyAsync(out, m->d_bout, n * (row + 16), hipMemcpyDeviceToHost, m->stream));
    SX_HIP(hipStreamSynchronize(m->stream));
    // status word of a chain: 0, 1 (domain error), or 2 + the index of its
    // first non-finite parameter; without a domain error the log density is
    // finite
    spread_rows(n, grad ? n * row : 0, [=](int64_t c) {
      double* o = out + c * (D + 2);
      const int64_t bad = checked ? first_non_finite(th + c * D, D) : -1;
      if (bad >= 0) o[D + 1] = 2.0 + static_cast<double>(bad);
      lp[b + c] = o[D + 1] == 0.0 ? o[0] : -INFINITY;
      if (grad && bad < 0) std::memcpy(grad + (b + c) * D, o + 1, row);
    });
    for (int64_t c = n - 1; c >= 0; --c)
      if (lp[b + c] == -INFINITY) {  // the last one's message
        const double status = out[c * (D + 2) + D + 1];
        worst = SX_EDOMAIN;
        set_error(status < 2.0 ? std::string(message)
                               : "log_prob: parameter " +
                                     std::to_string(static_cast<int64_t>(status - 2.0)) +
                                     " is not finite");
        break;
      }
  }
  queued.done = true;
  return worst;
}

// C chains of a logistic or normal context in FP64, evaluated together in
// slabs whose block partials stay within kSlabBytes.  Each chain's result is
// bitwise its single evaluation's.
constexpr size_t kSlabBytes = size_t(256) << 20;

int ensure_batch_partials(sx_glm* m, int64_t C) {
  if (m->bpart_cap >= C) return SX_OK;
  (void)hipFree(m->d_bpart);
  m->d_bpart = nullptr;
  m->bpart_cap = 0;
  SX_HIP(hipMalloc(&m->d_bpart, sizeof(double) * (m->K + 3) * m->blocks * C));
  m->bpart_cap = C;
  return SX_OK;
}

// One chain after the other, in the context's own buffers.
int one_by_one(sx_glm* m, const double* theta, int64_t C, int propto, int jacobian, double* lp,
               double* grad) {
  int worst = SX_OK;
  for (int64_t c = 0; c < C; ++c) {
    const int rc = eval(m, theta + c * m->D, propto, jacobian, lp + c,
                        grad ? grad + c * m->D : nullptr);
    if (rc == SX_EDOMAIN) {
      lp[c] = -INFINITY;
      worst = SX_EDOMAIN;
    } else if (rc) {
      return rc;
    }
  }
  return worst;
}

int fp64_batch(sx_glm* m, const double* theta, int64_t C, int propto, int jacobian, double* lp,
               double* grad) {
  SX_HIP(hipSetDevice(m->device));
  const int64_t E = m->K + 3;
  const int64_t fit = static_cast<int64_t>(kSlabBytes / (sizeof(double) * E * m->blocks));
  int64_t slab = std::max<int64_t>(1, std::min<int64_t>({C, fit, 1024}));
  // where the device has no room for the slab, half of it, and so on
  while (ensure_batch_partials(m, slab) != SX_OK || ensure_batch_staging(m, slab) != SX_OK) {
    (void)hipGetLastError();  // else the next launch's check reports it
    (void)hipFree(m->d_bpart);
    m->d_bpart = nullptr;
    m->bpart_cap = 0;
    if (slab == 1) return one_by_one(m, theta, C, propto, jacobian, lp, grad);
    slab = (slab + 1) / 2;
  }
  return batch_call(m, theta, C, slab, true, domain_message(m->family), lp, grad,
                    [=](int n) {
    return sx::plain_enqueue(m, m->d_btheta, m->d_bout, m->d_bpart, propto, jacobian, m->stream,
                             true, n);
  });
}

}  // namespace

extern "C" {

int sx_glm_logp_grad(sx_glm* m, const double* theta, int propto, int jacobian, double* lp,
                     double* grad) {
  return eval(m, theta, propto, jacobian, lp, grad);
}

int sx_glm_logp(sx_glm* m, const double* theta, int propto, int jacobian, double* lp) {
  return eval(m, theta, propto, jacobian, lp, nullptr);
}

int sx_glm_logp_grad_batch(sx_glm* m, const double* theta, int64_t C, int propto,
                           int jacobian, double* lp, double* grad) {
  if (!m || C < 0 || (C > 0 && (!theta || !lp))) {
    set_error("sx_glm_logp_grad_batch: invalid argument");
    return SX_EINVAL;
  }
  if (C == 0) return SX_OK;
  if (m->precision == SX_BF16X2 || m->family == SX_HIER_LOGIT) {
    const bool hier = m->family == SX_HIER_LOGIT;
    return batch_call(m, theta, C, C, false,
                      hier ? domain_message(m->family)
                           : "batched GLM: linear predictor or log density is not finite",
                      lp, grad, [=](int n) {
                        return hier ? sx::hier_enqueue(m, m->hw, m->d_btheta, n, m->d_bout, propto,
                                                       jacobian, m->precision == SX_FP32, m->stream)
                                    : sx::mx_enqueue(m, m->mx, m->d_btheta, n, m->d_bout, propto,
                                                     jacobian, m->stream);
                      });
  }
  return C > 1 ? fp64_batch(m, theta, C, propto, jacobian, lp, grad)
               : one_by_one(m, theta, C, propto, jacobian, lp, grad);
}

int sx_glm_time_logp_grad(sx_glm* m, const double* theta, int64_t C, int iters, int warmup,
                          double* ms_per_eval, double* ms_kernel) {
  if (!m || !theta || iters <= 0 || C < 1 ||
      (C > 1 && m->precision != SX_BF16X2 && m->family != SX_HIER_LOGIT)) {
    set_error("sx_glm_time_logp_grad: invalid argument");
    return SX_EINVAL;
  }
  SX_HIP(hipSetDevice(m->device));
  const size_t D = static_cast<size_t>(m->D);
  const bool batched = C > 1;
  if (batched) {
    int rc = ensure_batch_staging(m, C);
    if (rc) return rc;
    SX_HIP(hipMemcpy(m->d_btheta, theta, D * C * sizeof(double), hipMemcpyHostToDevice));
  } else {
    SX_HIP(hipMemcpy(m->d_theta, theta, D * sizeof(double), hipMemcpyHostToDevice));
  }
  auto one = [&](bool reduce) -> int {
    if (batched && m->family == SX_HIER_LOGIT)
      return sx::hier_enqueue(m, m->hw, m->d_btheta, static_cast<int>(C), m->d_bout, 1, 1,
                              m->precision == SX_FP32, m->stream);
    if (batched)
      return sx::mx_enqueue(m, m->mx, m->d_btheta, static_cast<int>(C), m->d_bout, 1, 1, m->stream);
    return enqueue_pass(m, 1, 1, reduce);
  };
  for (int i = 0; i < warmup; ++i) {
    int rc = one(true);
    if (rc) return rc;
  }
  SX_HIP(hipStreamSynchronize(m->stream));
  // full evaluations (for a single chain: bulk pass + cross-block reduction)
  SX_HIP(hipEventRecord(m->ev0, m->stream));
  for (int i = 0; i < iters; ++i) {
    int rc = one(true);
    if (rc) return rc;
  }
  SX_HIP(hipEventRecord(m->ev1, m->stream));
  SX_HIP(hipEventSynchronize(m->ev1));
  float ms = 0.f;
  SX_HIP(hipEventElapsedTime(&ms, m->ev0, m->ev1));
  if (ms_per_eval) *ms_per_eval = ms / iters;
  if (batched) {
    if (ms_kernel) *ms_kernel = ms / iters;
    return SX_OK;
  }
  // the bulk X pass alone (its partials are left unreduced)
  SX_HIP(hipEventRecord(m->ev0, m->stream));
  for (int i = 0; i < iters; ++i) {
    int rc = one(false);
    if (rc) return rc;
  }
  SX_HIP(hipEventRecord(m->ev1, m->stream));
  SX_HIP(hipEventSynchronize(m->ev1));
  SX_HIP(hipEventElapsedTime(&ms, m->ev0, m->ev1));
  if (ms_kernel) *ms_kernel = ms / iters;
  return SX_OK;
}

int sx_glm_kernel_config(const sx_glm* m, int* lanes_per_row, int* slots_per_lane,
                         int* blocks, int* threads, int* prefetch) {
  if (!m) {
    set_error("NULL model");
    return SX_EINVAL;
  }
  if (lanes_per_row) *lanes_per_row = m->geom.L;
  if (slots_per_lane) *slots_per_lane = m->geom.S;
  if (blocks) *blocks = m->blocks;
  if (threads) *threads = m->threads;
  if (prefetch) *prefetch = m->geom.prefetch;
  return SX_OK;
}

}  // extern "C"
