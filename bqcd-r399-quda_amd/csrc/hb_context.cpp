// hb_context.cpp - context lifecycle, staging buffers, error reporting.
#include <chrono>
#include <cstdarg>
#include <cstring>
#include <mutex>
#include <thread>

#include "hb_internal.h"

namespace hb {

static thread_local char g_err[1024] = "";

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
}

int ensure_dev_stage(Context *c, size_t bytes) {
  if (c->dev_stage_bytes >= bytes) return HB_OK;
  if (c->dev_stage) HB_HIP(hipFree(c->dev_stage));
  c->dev_stage = nullptr;
  c->dev_stage_bytes = 0;
  HB_HIP(device_alloc(c, &c->dev_stage, bytes));
  c->dev_stage_bytes = bytes;
  return HB_OK;
}

int ensure_host_stage(Context *c, size_t bytes) {
  if (c->host_stage_bytes >= bytes) return HB_OK;
  if (c->host_stage) HB_HIP(hipHostFree(c->host_stage));
  c->host_stage = nullptr;
  c->host_stage_bytes = 0;
  HB_HIP(hipHostMalloc(&c->host_stage, bytes, hipHostMallocDefault));
  c->host_stage_bytes = bytes;
  return HB_OK;
}

int wait_note(Context *c, int k, uint64_t seq, uint64_t *v) {
  using clock = std::chrono::steady_clock;
  // a query is not free for the kernels in flight: with one every 4096 pauses,
  // about 0.2 ms, block solves in FP32 took 0.3 to 0.7 % more (28^3x40, one right-hand
  // side 46.0 / 45.7 ms, four 164.9 / 164.4; 32^3x48, one 78.2 / 77.8)
  constexpr auto kQuery = std::chrono::milliseconds(50);
  clock::time_point due{};
  for (unsigned spin = 1;; spin++) {
    *v = __atomic_load_n(c->note + k, __ATOMIC_ACQUIRE);
    if (*v >> 2 >= seq) return HB_OK;
    __builtin_ia32_pause();
    if (spin % 4096) continue;
    std::this_thread::yield();  // there may be more threads with a context than cores
    const clock::time_point now = clock::now();
    if (due == clock::time_point{}) due = now + kQuery;
    if (now < due) continue;
    due = now + kQuery;
    // every report has been written once the stream is empty: the wait ends
    // there also when a kernel failed
    const hipError_t e = hipStreamQuery(c->stream);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    HB_HIP(e);
    *v = __atomic_load_n(c->note + k, __ATOMIC_ACQUIRE);
    HB_CHECK(*v >> 2 >= seq, HB_E_HIP, "a solve's progress was not reported");
    return HB_OK;
  }
}

int Watch::look(int *flag) {
  const uint64_t last = c_->note_seq;
  uint64_t v = 0;
  HB_TRY(wait_note(c_, 0, last - 1, &v));
  const bool set = (v & 3) != 0, follows = v >> 2 < last || set_;
  set_ = set && !follows;
  *flag = set && follows ? (int)(v & 3) : 0;
  return HB_OK;
}

static bool release_spare(Context *c) {
  if (!c->spare.p) return false;
  (void)hipFree(c->spare.p);
  c->spare = Field{};
  return true;
}

hipError_t device_alloc_bytes(Context *c, void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipErrorOutOfMemory || !release_spare(c)) return e;
  (void)hipGetLastError();
  return hipMalloc(p, bytes);
}

void *spare(Context *c, size_t bytes) {
  if (c->spare.bytes >= bytes) return c->spare.p;
  release_spare(c);
  size_t free = 0, total = 0;
  if (hipMemGetInfo(&free, &total) != hipSuccess || free < bytes + total / 4 ||
      hipMalloc(&c->spare.p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    c->spare = Field{};
    return nullptr;
  }
  c->spare.bytes = bytes;
  return c->spare.p;
}

// Scratch slots grow on demand and are kept for the life of the context.
void *scratch(Context *c, int slot, size_t bytes, int *rc) {
  *rc = HB_OK;
  if ((int)c->scratch.size() <= slot) c->scratch.resize(slot + 1);
  Field &f = c->scratch[slot];
  if (f.bytes >= bytes) return f.p;
  if (f.p) {
    hipError_t e = hipFree(f.p);
    if (e != hipSuccess) {
      set_error("hipFree(scratch): %s", hipGetErrorString(e));
      *rc = HB_E_HIP;
      return nullptr;
    }
  }
  f.p = nullptr;
  f.bytes = 0;
  hipError_t e = device_alloc(c, &f.p, bytes);
  if (e != hipSuccess) {
    set_error("hipMalloc(scratch %zu bytes): %s", bytes, hipGetErrorString(e));
    *rc = HB_E_NOMEM;
    return nullptr;
  }
  f.bytes = bytes;
  return f.p;
}

}  // namespace hb

using namespace hb;

extern "C" {

const char *hb_last_error(void) { return g_err; }

int hb_init(const int L[4], const int bc[4], int device, hb_context **out) {
  HB_CHECK(L && bc && out, HB_E_ARG, "hb_init: null argument");
  for (int m = 0; m < 4; m++) {
    HB_CHECK(L[m] >= 2 && (L[m] % 2) == 0, HB_E_ARG, "hb_init: L[%d]=%d must be even and >= 2",
             m, L[m]);
    HB_CHECK(bc[m] == 1 || bc[m] == -1, HB_E_ARG, "hb_init: bc[%d]=%d must be +1 or -1", m,
             bc[m]);
  }
  long long vol = (long long)L[0] * L[1] * L[2] * L[3];
  // every field is addressed through buffer resources with 32-bit byte
  // offsets; the largest single-buffer field is an FP64 spinor (192 B per site)
  HB_CHECK(192LL * (vol / 2) < (1LL << 32), HB_E_ARG,
           "hb_init: lattice too large (%lld sites per parity; an FP64 spinor field must stay below 4 GiB)",
           (long long)(vol / 2));
  int ndev = 0;
  HB_HIP(hipGetDeviceCount(&ndev));
  HB_CHECK(device >= 0 && device < ndev, HB_E_ARG, "hb_init: device %d of %d", device, ndev);
  HB_HIP(hipSetDevice(device));
  Context *c = new Context();
  for (int m = 0; m < 4; m++) {
    c->g.L[m] = L[m];
    c->g.bc[m] = bc[m];
  }
  c->g.nxh = L[0] / 2;
  c->g.vh = (int)(vol / 2);
  c->device = device;
  // a blocking stream: ordered with the null stream, so a caller that works on
  // the null stream (and passes no stream of its own) needs no extra waits
  hipError_t e = hipStreamCreate(&c->own_stream);
  if (e != hipSuccess) {
    delete c;
    set_error("hipStreamCreate: %s", hipGetErrorString(e));
    return HB_E_HIP;
  }
  c->stream = c->own_stream;
  noalloc_setup(device);
  // reduction partials: up to 16 values per block of a site-parallel grid
  c->red_blocks = nblocks(2 * c->g.vh) + 64;
  e = hipMalloc(&c->red, sizeof(double) * 16 * (size_t)c->red_blocks);
  // the host reads the notes while the kernels that write them are in flight, so
  // the words must be coherent whatever the runtime's default is (HIP_HOST_COHERENT)
  if (e == hipSuccess)
    e = hipHostMalloc(reinterpret_cast<void **>(&c->note), kNotes * sizeof(uint64_t), hipHostMallocCoherent);
  if (e != hipSuccess) {
    set_error("hb_init: %s", hipGetErrorString(e));
    hb_finalize(reinterpret_cast<hb_context *>(c));
    return HB_E_HIP;
  }
  std::memset(c->note, 0, kNotes * sizeof(uint64_t));
  *out = reinterpret_cast<hb_context *>(c);
  return HB_OK;
}

int hb_finalize(hb_context *ctx) {
  Context *c = reinterpret_cast<Context *>(ctx);
  if (!c) return HB_OK;
  // teardown: errors are ignored, every resource is released regardless
  (void)hipSetDevice(c->device);
  if (c->own_stream) (void)hipStreamSynchronize(c->own_stream);
  (void)hipFree(c->gauge);
  for (auto *p : c->clov) (void)hipFree(p);
  (void)hipFree(c->gauge64r);
  (void)hipFree(c->gauge32);
  for (auto *p : c->clov32) (void)hipFree(p);
  (void)hipFree(c->gauge16);
  for (auto *p : c->clov16) (void)hipFree(p);
  for (auto &f : c->scratch) (void)hipFree(f.p);
  (void)hipFree(c->spare.p);
  (void)hipFree(c->red);
  (void)hipFree(c->dev_stage);
  if (c->host_stage) (void)hipHostFree(c->host_stage);
  if (c->note) (void)hipHostFree(c->note);
  if (c->own_stream) (void)hipStreamDestroy(c->own_stream);
  delete c;
  return HB_OK;
}

int hb_volh(const hb_context *ctx) {
  const Context *c = reinterpret_cast<const Context *>(ctx);
  return c ? c->g.vh : 0;
}

int hb_set_stream(hb_context *ctx, void *stream) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_CHECK(c, HB_E_ARG, "hb_set_stream: null context");
  c->stream = stream ? static_cast<hipStream_t>(stream) : c->own_stream;
  return HB_OK;
}

int hb_set_link_recon(hb_context *ctx, int recon) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_CHECK(c, HB_E_ARG, "hb_set_link_recon: null context");
  HB_CHECK(recon == 12 || recon == 18, HB_E_ARG, "hb_set_link_recon: %d (use 12 or 18)", recon);
  c->link_recon = recon;
  return HB_OK;
}

int hb_multi_block_size(hb_context *ctx) {
  Context *c = reinterpret_cast<Context *>(ctx);
  return c ? c->last_block : 0;
}

int hb_multi_block_limit(int volh, int precision) {
  if (volh < 1 || (precision != HB_PREC_F32 && precision != HB_PREC_F16)) return 0;
  static const int cand[5] = {12, 8, 4, 2, 1};
  for (int nr : cand)
    if (hb::multi_block_fits(volh, nr, precision)) return nr;
  return 0;
}

int hb_multi_tile(hb_context *ctx) {
  Context *c = reinterpret_cast<Context *>(ctx);
  return c ? c->last_tile : 0;
}

int hb_multi_set_tile(hb_context *ctx, int tile) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_CHECK(c, HB_E_ARG, "hb_multi_set_tile: null context");
  HB_CHECK(tile == 128 || tile == 256, HB_E_ARG, "hb_multi_set_tile: tile %d (use 128 or 256)", tile);
  c->user_tile = tile;
  return HB_OK;
}

int hb_last_timing(hb_context *ctx, double *solve_ms, int *n_matvec) {
  Context *c = reinterpret_cast<Context *>(ctx);
  HB_CHECK(c, HB_E_ARG, "hb_last_timing: null context");
  if (solve_ms) *solve_ms = c->last_solve_ms;
  if (n_matvec) *n_matvec = c->last_n_matvec;
  return HB_OK;
}

}  // extern "C"
