// CPU driver of the large host copies (fsibe_2d_amd/csrc/transfer.hpp) on
// stand-ins for the HIP calls that it makes: "device" memory is ordinary
// memory and a copy is over when it is issued.  argv[1] names the case; prints
// one line, and the exit status is 0 where the case holds.
#include <signal.h>
#include <sys/wait.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <string>

#include "../../fsibe_2d_amd/csrc/transfer.hpp"

// ---- stand-ins -------------------------------------------------------------
static void (*on_query)() = nullptr;  // called once, by the next event query
static int copies = 0;                // hipMemcpyAsync calls
extern "C" {
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
  ++copies;
  memcpy(dst, src, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorInvalidValue; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) {
  if (on_query) {
    auto f = on_query;
    on_query = nullptr;
    f();
  }
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}

// ---- cases -----------------------------------------------------------------
// bytes of 'device' -> host -> 'device', at an odd host address
static bool round_trip(size_t n) {
  std::vector<unsigned char> dev(n), host(n + 1, 0), back(n, 0);
  unsigned x = 12345u + (unsigned)n;
  for (auto &b : dev) b = (unsigned char)((x = x * 1664525u + 1013904223u) >> 24);
  auto &t = fsibe::Transfer::get();
  return t.download(host.data() + 1, dev.data(), n, nullptr) == hipSuccess &&
         t.upload(back.data(), host.data() + 1, n, nullptr) == hipSuccess && back == dev;
}

// the child's exit status, or -1 if it has not ended within 20 s (it is then killed)
static int wait_child(pid_t p) {
  for (int k = 0; k < 2000; ++k) {
    int st = 0;
    if (waitpid(p, &st, WNOHANG) == p) return WIFEXITED(st) ? WEXITSTATUS(st) : 256;
    std::this_thread::sleep_for(std::chrono::milliseconds(10));
  }
  kill(p, SIGKILL);
  waitpid(p, nullptr, 0);
  return -1;
}

static pid_t child = 0;
static void fork_inside_a_copy() {
  child = fork();
  if (child == 0) exit(7);
}

// destroyed after everything that a first copy makes: copies once more then
struct Late {
  bool on = false;
  ~Late() {
    if (on && !round_trip(9u << 20)) _exit(1);
  }
};
static Late late;

int main(int argc, char **argv) {
  const std::string c = argc > 1 ? argv[1] : "";
  constexpr size_t kBig = (size_t)9 << 20;
  if (c == "sizes") {
    const size_t d = (size_t)8 << 20, u = (size_t)48 << 20;
    for (size_t n : {(size_t)1, d - 1, d, d + 1, kBig + 3, u - 1, u, u + 1, (size_t)70 << 20})
      if (!round_trip(n)) return std::printf("%zu bytes differ\n", n), 1;
    std::puts("equal");
    return 0;
  }
  if (c == "lines") {  // the runtime's path (one copy) below each direction's line, chunks from there on
    std::vector<char> a((size_t)48 << 20), b(a.size());
    auto count = [&](bool up, size_t n) {
      copies = 0;
      auto &t = fsibe::Transfer::get();
      (void)(up ? t.upload(a.data(), b.data(), n, nullptr) : t.download(a.data(), b.data(), n, nullptr));
      return copies;
    };
    const size_t d = (size_t)8 << 20, u = a.size();
    const bool ok = count(false, (size_t)6 << 20) == 1 && count(false, d - 1) == 1 && count(false, d) > 1 &&
                    count(true, d) == 1 && count(true, (size_t)32 << 20) == 1 && count(true, u - 1) == 1 && count(true, u) > 1;
    std::puts(ok ? "as measured" : "another line");
    return ok ? 0 : 1;
  }
  if (c == "late") {
    late.on = true;
    if (!round_trip(kBig)) return 1;
    std::puts("copied");
    std::fflush(stdout);
    return 0;  // Late's destructor copies
  }
  int want = 0;
  if (c == "fork") {  // after a copy; the child copies too, then ends normally
    if (!round_trip(kBig)) return 1;
    child = fork();
    if (child == 0) exit(round_trip(kBig) ? 0 : 1);
  } else if (c == "fork_inside") {  // from the copying thread, while the helpers work
    on_query = fork_inside_a_copy;
    if (!round_trip(kBig)) return 1;
    want = 7;
  } else {
    return 2;
  }
  const int st = wait_child(child);
  std::printf("child %d\n", st);
  return st == want && round_trip(kBig) ? 0 : 1;
}
