// host_check.hip -- host-only check of the library's planning code under
// AddressSanitizer / UndefinedBehaviorSanitizer (built by `make host-check`
// with --offload-host-only: no device code, no GPU needed, nothing launched).
//
// Every backward composition is run in its sizing mode (the same dispatch as
// a real call: algorithm choice, stride phases, weight-gradient plans,
// split-K plans, im2col sizes; it stops before any launch) over a grid of
// shapes, dtypes and algorithms, together with the plans of products and Linear
// layers up to the largest sizes, of convolutions over channels-last copies (and that
// their addresses stay within the copies), the growth of a stream's workspace over a played
// device, the algorithm selectors and the shape checks of the
// entry points.  A sanitizer report, a bad size or a bad plan fails.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

// The allocator and the stream queries behind the workspaces, played by the host: a
// device of `room` bytes whose calls are written down in order (m, s, f).
namespace fake {
size_t room = SIZE_MAX;
bool capturing = false;
hipError_t sync = hipSuccess;
std::vector<char> calls;
hipError_t alloc(void** p, size_t bytes) {
  calls.push_back('m');
  if (bytes > room) return hipErrorOutOfMemory;
  *p = malloc(bytes);
  return hipSuccess;
}
hipError_t release(void* p) {
  calls.push_back('f');
  free(p);
  return hipSuccess;
}
hipError_t synchronize(hipStream_t) {
  calls.push_back('s');
  return sync;
}
hipError_t is_capturing(hipStream_t, hipStreamCaptureStatus* s) {
  *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
}  // namespace fake
#define hipMalloc fake::alloc
#define hipFree fake::release
#define hipStreamSynchronize fake::synchronize
#define hipStreamIsCapturing fake::is_capturing
#include "vh_api.hip"

namespace {
using namespace vh;
long n = 0, fails = 0;

void expect(bool ok, const char* what) {
  ++n;
  if (!ok) {
    printf("workspace: %s\n", what);
    ++fails;
  }
}
bool called(const char* seq) {
  const bool same = std::string(fake::calls.begin(), fake::calls.end()) == seq;
  fake::calls.clear();
  return same;
}

// Growth of a stream's workspace: an optional request that cannot be had changes nothing.
void check_workspace() {
  const hipStream_t st = reinterpret_cast<hipStream_t>(64), st2 = reinterpret_cast<hipStream_t>(128);
  void *a, *b;
  expect(ws_get(st, 1000, &a) == VH_OK && a && called("m"), "first request");
  fake::room = 1 << 20;
  set_error(VH_OK, "before");
  expect(ws_optional(st, 2 << 20, &b) == VH_ERR_OOM && !b && called("m"), "optional request without memory");
  expect(falls_back(VH_ERR_OOM) && !strcmp(g_err, "before"), "an error was left by a call that falls back");
  expect(ws_get(st, 1000, &b) == VH_OK && b == a && called(""), "the old buffer is gone");
  expect(ws_optional(st, 2 << 20, &b) == VH_ERR_OOM && called(""), "a second try right away");
  expect(ws_optional(st, 3000, &b) == VH_OK && b != a && called("msf"), "a smaller optional request; new buffer before the old goes");
  fake::room = 2 << 20;
  for (int i = 0; i < kRefusals; ++i) {
    fake::room = SIZE_MAX;
    if (ws_optional(st, 2 << 20, &b) == VH_OK) break;
  }
  expect(ws_optional(st, 2 << 20, &b) == VH_OK && b, "tried again once there is memory");
  fake::calls.clear();
  // capture: never grows; what is there serves, and is retired when outgrown
  fake::capturing = true;
  set_error(VH_OK, "before");
  expect(ws_optional(st, 8 << 20, &a) == VH_ERR_CAPTURE && !a && !strcmp(g_err, "before") && called(""), "optional growth in a capture");
  expect(ws_get(st, 1000, &a) == VH_OK && a == b && called(""), "use in a capture");
  expect(ws_get(st, 8 << 20, &a) == VH_ERR_CAPTURE && called(""), "growth in a capture");
  fake::capturing = false;
  const size_t retired = g_ws_retired.size();
  expect(ws_optional(st, 8 << 20, &a) == VH_OK && called("m") && g_ws_retired.size() == retired + 1, "a captured buffer is retired");
  // a required request frees first; a failed synchronisation is the call's own error
  expect(ws_get(st, 16 << 20, &a) == VH_OK && called("sfm"), "required growth");
  fake::sync = hipErrorLaunchFailure;
  expect(ws_optional(st, 32 << 20, &a) == VH_ERR_LAUNCH && !falls_back(VH_ERR_LAUNCH), "a failed synchronisation");
  fake::sync = hipSuccess;
  fake::calls.clear();
  // the fixed scratch
  char scr[64];
  {
    FixedWs guard(scr, sizeof(scr));
    set_error(VH_OK, "before");
    expect(ws_optional(st2, 65, &a) == VH_ERR_UNSUPPORTED && !strcmp(g_err, "before"), "optional beyond the scratch");
    expect(ws_optional(st2, 64, &a) == VH_OK && a == scr && called(""), "the scratch");
  }
}

// The plan of a product or a Linear layer's pair: the splits cover K, the workspace
// holds them, and no block is left with a long K of its own beside an idle chip.
void check_mm(int dt, const DenseProblem* p, int np) {
  MmInfo o;
  ++n;
  if (!mm_info(dt, p, np, &o)) return;
  const long bk = dt == VH_BF16 ? 64 : 32;
  double work = 0;
  size_t part = 0;
  for (int i = 0; i < np; ++i) {
    const long st = (p[i].K + bk - 1) / bk;
    work += (double)((p[i].M + o.bm - 1L) / o.bm) * ((p[i].N + o.bn - 1L) / o.bn) * st;
    if (o.splits[i] > 1) part += (size_t)o.splits[i] * p[i].M * p[i].N * 4;
    if (o.splits[i] < 1 || (long)o.splits[i] * o.per[i] < st || (long)(o.splits[i] - 1) * o.per[i] >= st) {
      printf("bad splits %d x %d of %ld stages: %d %d %d\n", o.splits[i], o.per[i], st, p[i].M, p[i].N, p[i].K);
      ++fails;
    }
  }
  for (int i = 0; i < np; ++i)
    if (o.per[i] > 64 + 3 * work / 256) {
      printf("a block of %d stages, %.0f a CU: dt%d np%d %d %d %d\n", o.per[i], work / 256, dt, np, p[i].M, p[i].N, p[i].K);
      ++fails;
    }
  if (o.bytes < part) {
    printf("workspace %zu below the partials %zu: %d %d %d\n", o.bytes, part, p[0].M, p[0].N, p[0].K);
    ++fails;
  }
}

void check_products() {
  char* q = reinterpret_cast<char*>(4096);
  const int dims[] = {1, 2, 7, 10, 31, 64, 65, 130, 500, 513, 1000, 2048, 4097, 16384, 100003, 1 << 24, (1 << 30) + 1, INT32_MAX};
  for (int dt : {(int)VH_F32, (int)VH_BF16})
    for (int M : dims)
      for (int N : dims)
        for (int K : dims) {
          if (std::max({(long)M * K, (long)K * N, (long)M * N}) > kMaxElems) continue;
          const DenseProblem nn{q, K, false, q, N, true, q, N, M, N, K, nullptr}, nt{q, K, false, q, K, false, q, N, M, N, K, nullptr},
              tn{q, M, true, q, N, true, q, N, M, N, K, nullptr};
          check_mm(dt, &nn, 1);
          check_mm(dt, &nt, 1);
          check_mm(dt, &tn, 1);
          // a Linear layer of M rows, K -> N features
          const DenseProblem pair[2] = {{q, N, false, q, N, false, q, K, M, K, N, nullptr}, {q, K, true, q, N, true, q, N, K, N, M, q}};
          check_mm(dt, pair, 2);
          (void)linear_pair(dt, pair);
        }
}
// A convolution's plans over channels-last copies: forward, both gradients apart and together.
void check_gather(int dt, const ConvDims& d) {
  char* q = reinterpret_cast<char*>(4096);
  GatherCall y{}, dx{}, dw{}, both{};
  y.g = dx.g = dw.g = both.g = geom_of(d);
  y.x = y.w = dx.dy = dx.w = dw.x = dw.dy = both.x = both.dy = both.w = q;
  y.y = dx.dx = dw.dw = dw.db = both.dx = both.dw = q;
  for (const GatherCall* c : {&y, &dx, &dw, &both}) {
    GatherInfo o;
    ++n;
    if (!gather_info(dt, *c, &o)) continue;
    if (!o.ok || o.bytes != gather_ws(dt, *c) || o.bytes > kGatherMostWs || o.images < 1 || o.images > d.B) {
      printf("channels-last plan: dt%d B%ld C%ld O%ld %ldx%ld K%ldx%ld S%ldx%ld P%ldx%ld: %d images, %zu bytes, ok %d\n", dt, d.B,
             d.C, d.O, d.H, d.W, d.KH, d.KW, d.SH, d.SW, d.PH, d.PW, o.images, o.bytes, (int)o.ok);
      ++fails;
    }
  }
}

void check_gathers() {
  const long Bs[] = {1, 3, 64, 1000}, Cs[] = {1, 7, 64, 513}, Hs[] = {1, 2, 9, 57, 300}, Ks[] = {1, 2, 3, 8};
  for (int dt : {(int)VH_F32, (int)VH_BF16})
    for (long B : Bs)
      for (long C : Cs)
        for (long O : Cs)
          for (long H : Hs)
            for (long W : Hs)
              for (long K : Ks)
                for (long S : {1L, 2L, 3L, 5L})
                  for (long P : {0L, 1L, K, 40L}) {
                    ConvDims d{B, C, O, H, W, K, std::min(K, 3L), S, S > 3 ? 1 : S, P, P / 2, 0, 0};
                    if (H + 2 * d.PH < d.KH || W + 2 * d.PW < d.KW) continue;
                    d.HO = (H + 2 * d.PH - d.KH) / d.SH + 1;
                    d.WO = (W + 2 * d.PW - d.KW) / d.SW + 1;
                    if (check_conv(d, true) == VH_OK) check_gather(dt, d);
                  }
  // padding beyond what 32 bits hold when doubled
  const ConvDims wide{1, 1, 1, INT32_MAX, 1, 1, 1, 1, 1, 0, 0, INT32_MAX, 1}, pad{1, 1, 1, 1, 1, 3, 3, 1 << 29, 1 << 29, 1 << 30, 1 << 30, 4, 4};
  for (int dt : {(int)VH_F32, (int)VH_BF16}) {
    check_gather(dt, wide);
    check_gather(dt, pad);
  }
  // tiles that tests/test_gpu_gather.py is after (bf16)
  const struct {
    long B, C, O, H, W, K, S;
    int bm, bn, ks;
  } tiles[] = {{16, 120, 130, 21, 23, 3, 1, 64, 64, 2},  {5, 120, 250, 33, 31, 3, 1, 64, 64, 2},  {64, 60, 64, 39, 41, 1, 2, 64, 64, 1},
               {64, 300, 64, 39, 41, 1, 2, 64, 64, 1},   {128, 60, 64, 39, 41, 1, 2, 64, 128, 1}, {128, 250, 64, 39, 41, 1, 2, 64, 128, 1},
               {96, 100, 120, 29, 31, 3, 1, 128, 128, 1}, {2, 250, 40, 13, 11, 3, 1, 32, 32, 4},  {4, 40, 100, 27, 29, 3, 1, 32, 64, 2}};
  for (const auto& t : tiles) {
    const long HO = (t.H + (t.K / 2) * 2 - t.K) / t.S + 1, WO = (t.W + (t.K / 2) * 2 - t.K) / t.S + 1;
    const ConvDims d{t.B, t.C, t.O, t.H, t.W, t.K, t.K, t.S, t.S, t.K / 2, t.K / 2, HO, WO};
    GatherCall c{};
    c.g = geom_of(d);
    c.x = c.w = c.y = const_cast<char*>("");
    GatherInfo o;
    ++n;
    if (!gather_info(VH_BF16, c, &o) || o.bm != t.bm || o.bn != t.bn || o.ks != t.ks) {
      printf("tile of B%ld C%ld O%ld %ldx%ld: %d x %d, %d groups\n", t.B, t.C, t.O, t.H, t.W, o.bm, o.bn, o.ks);
      ++fails;
    }
  }
}

// The narrow fp32 layers take the faster of their two paths, pass by pass, where one
// was measured 8 % ahead (us: halo, channels-last).
void check_halo_rule() {
  const struct {
    HaloPass pass;
    long C, B, H, W;
    float halo, copies;
  } rows[] = {
      {HALO_TO_64, 32, 16, 28, 28, 21.4f, 15.8f},  {HALO_TO_64, 32, 64, 28, 28, 23.4f, 33.0f},  {HALO_TO_64, 32, 71, 28, 28, 41.8f, 33.8f},
      {HALO_TO_64, 32, 110, 28, 28, 42.4f, 49.4f}, {HALO_TO_64, 32, 200, 28, 28, 82.9f, 70.3f}, {HALO_TO_64, 32, 64, 8, 8, 20.9f, 11.9f},
      {HALO_TO_64, 32, 96, 20, 20, 41.5f, 27.9f},  {HALO_TO_32, 64, 32, 28, 28, 22.3f, 24.4f},  {HALO_TO_32, 64, 16, 28, 28, 21.7f, 16.7f},
      {HALO_TO_32, 64, 96, 28, 28, 42.3f, 47.7f},  {HALO_TO_32, 64, 110, 28, 28, 42.6f, 47.0f}, {HALO_TO_32, 64, 256, 28, 28, 87.3f, 96.8f},
      {HALO_TO_32, 64, 128, 20, 20, 41.9f, 38.5f}, {HALO_WGRAD, 32, 64, 28, 28, 28.8f, 40.7f},  {HALO_WGRAD, 32, 8, 28, 28, 22.4f, 18.1f},
      {HALO_WGRAD, 32, 256, 28, 28, 99.5f, 113.f}, {HALO_WGRAD, 32, 110, 28, 28, 50.6f, 58.1f}, {HALO_WGRAD, 32, 512, 28, 28, 192.f, 216.f},
      {HALO_WGRAD, 64, 16, 28, 28, 24.3f, 26.8f},  {HALO_WGRAD, 64, 71, 28, 28, 47.4f, 56.7f},  {HALO_WGRAD, 64, 200, 28, 28, 95.f, 134.8f},
      {HALO_WGRAD, 64, 256, 28, 20, 97.5f, 123.f}, {HALO_WGRAD, 64, 128, 8, 8, 31.2f, 21.7f},   {HALO_WGRAD, 64, 512, 20, 20, 140.f, 173.f},
  };
  for (const auto& r : rows) {
    const ConvDims d{r.B, r.C, 96 - r.C, r.H, r.W, 3, 3, 1, 1, 1, 1, r.H, r.W};
    ++n;
    if (halo_f32_pays(d, r.pass, false, false) != (r.halo < r.copies)) {
      printf("narrow fp32 layer, pass %d, %ld channels, %ld x %ld x %ld: the slower path\n", r.pass, r.C, r.B, r.H, r.W);
      ++fails;
    }
  }
  // both gradients of 32 -> 64 channels @14x12, 96 images: 40.4 us over shared copies, 47.1 apart
  const ConvDims d{96, 32, 64, 14, 12, 3, 3, 1, 1, 1, 1, 14, 12};
  if (halo_f32_pays(d, HALO_TO_32, true, false) || halo_f32_pays(d, HALO_WGRAD, false, true)) {
    printf("narrow fp32 layer: gradients apart that share their copies\n");
    ++fails;
  }
}
// fp32 layers of few positions: M, positions, channels, taps; us generic, channels-last.
void check_few_positions() {
  const struct {
    long M, pos, C, RS;
    float generic, copies;
  } rows[] = {{60, 32, 778, 25, 26.3f, 136.f}, {33, 162, 459, 9, 18.7f, 35.4f},   {512, 49, 512, 9, 33.7f, 47.f},  {256, 49, 256, 9, 21.9f, 25.7f}, {16, 784, 256, 9, 13.9f, 25.f}, {48, 432, 192, 9, 16.5f, 20.7f}, {192, 224, 64, 25, 22.6f, 21.3f}, {2, 1250, 128, 16, 14.1f, 20.7f},  {72, 225, 468, 16, 24.5f, 59.5f},
              {577, 98, 453, 16, 43.5f, 65.2f}, {108, 1053, 940, 9, 47.6f, 68.7f}, {60, 1734, 625, 25, 103.f, 112.f}, {333, 343, 721, 9, 63.1f, 56.8f}, {228, 768, 618, 25, 157.f, 112.f},
              {512, 392, 512, 9, 53.1f, 48.2f}, {164, 256, 192, 9, 22.8f, 21.f},   {199, 125, 240, 9, 28.7f, 25.3f},  {68, 936, 170, 9, 21.8f, 19.8f}};
  for (const auto& r : rows) {
    ++n;
    if (copies_pay(VH_F32, r.M, r.pos, r.C, r.RS) != (r.copies < r.generic)) {
      printf("fp32 %ld x %ld, %ld channels, %ld taps: the slower path\n", r.M, r.pos, r.C, r.RS);
      ++fails;
    }
  }
}

// fp32 1x1 layers: the path measured as the faster for a forward of M rows
void check_pointwise() {
  const struct {
    long M, K, B, H, S;
    float generic, copies;
  } rows[] = {{64, 256, 64, 56, 1, 97.8f, 156.7f}, {64, 64, 32, 56, 1, 25.3f, 29.6f},    {16, 64, 32, 56, 1, 20.9f, 23.3f},
              {16, 64, 64, 56, 1, 39.4f, 36.9f},   {48, 64, 100, 13, 1, 12.0f, 13.3f},   {128, 64, 64, 56, 1, 87.1f, 71.1f},
              {64, 128, 16, 14, 1, 13.7f, 10.1f},  {48, 160, 12, 56, 1, 22.0f, 27.0f},   {64, 256, 16, 112, 2, 36.5f, 111.5f},
              {256, 64, 32, 56, 2, 26.6f, 29.9f},  {512, 128, 16, 112, 2, 131.6f, 124.5f}, {64, 64, 32, 28, 2, 11.0f, 10.6f}};
  for (const auto& r : rows) {
    const long HO = (r.H - 1) / r.S + 1;
    const ConvDims d{r.B, r.K, r.M, r.H, r.H, 1, 1, r.S, r.S, 0, 0, HO, HO};
    ++n;
    if (pointwise_once(VH_F32, d, r.M, true) != (r.generic < r.copies)) {
      printf("fp32 1x1 %ld -> %ld, %ld images of %ld, stride %ld: the slower path\n", r.K, r.M, r.B, r.H, r.S);
      ++fails;
    }
  }
}
}  // namespace

int main() {
  const long Bs[] = {1, 2, 3, 16, 128};
  const long Cs[] = {1, 3, 16, 27, 64, 256};
  const long Hs[] = {1, 5, 14, 28, 56, 256};
  const long Ks[] = {1, 3, 5, 7};
  const long Ss[] = {1, 2, 3, 4, 5};
  char dummy[64];
  const void* p = dummy;
  for (long B : Bs)
    for (long C : Cs)
      for (long O : Cs)
        for (long H : Hs)
          for (long K : Ks)
            for (long S : Ss)
              for (long P = 0; P <= K; P += (K > 2 ? K / 2 : 1)) {
                if (B * C * H * H > (1L << 26) || B * O * H * H > (1L << 26)) continue;
                for (int dt : {(int)VH_F32, (int)VH_BF16})
                  for (int algo : {(int)VH_ALGO_DIRECT, (int)VH_ALGO_IM2COL, (int)VH_ALGO_IGEMM}) {
                    size_t need = (size_t)-1;
                    const int st = conv2d_backward_impl(dt, algo, p, p, p, (void*)p, (void*)p, (void*)p, B, C, O,
                                                        H, H, K, K, S, S, P, P, nullptr, false, &need);
                    ++n;
                    // valid geometry must plan (sizes below 2^31 elements); invalid must be rejected
                    const bool geom_ok = H + 2 * P >= K;
                    if (geom_ok && st != VH_OK && st != VH_ERR_UNSUPPORTED) {
                      printf("unexpected status %d: B%ld C%ld O%ld H%ld K%ld S%ld P%ld dt%d algo%d: %s\n", st, B, C,
                             O, H, K, S, P, dt, algo, g_err);
                      ++fails;
                    }
                    if (!geom_ok && st == VH_OK) {
                      printf("accepted bad geometry B%ld C%ld H%ld K%ld P%ld\n", B, C, H, K, P);
                      ++fails;
                    }
                    if (st == VH_OK && need == (size_t)-1) {
                      printf("no size: B%ld C%ld O%ld H%ld K%ld S%ld P%ld\n", B, C, O, H, K, S, P);
                      ++fails;
                    }
                  }
                (void)vh_conv_algo_auto_select(B, C, H, H, K, 1);
                (void)vh_conv_algo_auto_select(B, C, H, H, K, 0);
                (void)vh_conv_algo_select_mi355x(B, C, O, H, H, K, K, S, S, P, P);
              }
  // shape checks of the entry points' validation (negative, zero, overflow)
  ConvDims bad[] = {{-1, 1, 1, 4, 4, 3, 3, 1, 1, 1, 1, 4, 4},
                    {1, 0, 1, 4, 4, 3, 3, 1, 1, 1, 1, 4, 4},
                    {1, 1, 1, 4, 4, 3, 3, 0, 1, 1, 1, 4, 4},
                    {1, 1, 1, 4, 4, 3, 3, 1, 1, -1, 1, 4, 4},
                    {1, 1, 1, 4, 4, 3, 3, 1, 1, 1, 1, 5, 4},
                    {1L << 20, 1L << 10, 1, 64, 64, 3, 3, 1, 1, 1, 1, 64, 64}};
  for (const ConvDims& d : bad) {
    ++n;
    if (check_conv(d, true) == VH_OK) {
      printf("check_conv accepted a bad shape (B%ld C%ld SH%ld PH%ld HO%ld)\n", d.B, d.C, d.SH, d.PH, d.HO);
      ++fails;
    }
  }
  check_workspace();
  check_gathers();
  check_products();
  check_halo_rule();
  check_few_positions();
  check_pointwise();
  printf("host_check: %ld plans, %ld failures\n", n, fails);
  return fails ? 1 : 0;
}
