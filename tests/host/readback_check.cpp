// Host check of the pinned read-back (mh_readback.h) over stand-ins of the HIP calls.  The argument
// names the check; prints the reads made and the bytes that came out wrong.
#define MH_BLOCK 256
#include "../../mahyco_amd/csrc/mh_readback.h"

#include <cstdio>
#include <string>
#include <vector>

static std::vector<char> field(size_t n, unsigned seed) {
  std::vector<char> f(n);
  unsigned x = seed * 2654435761u + 1u;
  for (auto& b : f) {
    x = x * 1664525u + 1013904223u;
    b = (char)(x >> 24);
  }
  return f;
}
// one read of field f through the stage, as a copy enqueued slot by slot; the bytes that differ
static long read_field(HostStage& stage, StubStream& stream, const std::vector<char>& f) {
  std::vector<char> out(f.size());
  const hipError_t e = read_back(stage, &stream, out.data(), f.size(), [&](char* pin, size_t off, size_t len) {
    std::memcpy(pin, f.data() + off, len);
    std::this_thread::yield();
    return hipSuccess;
  });
  if (e != hipSuccess) return (long)f.size();
  long bad = 0;
  for (size_t i = 0; i < f.size(); ++i) bad += out[i] != f[i];
  return bad;
}

int main(int argc, char** argv) {
  const std::string check = argc > 1 ? argv[1] : "";
  long reads = 0;
  std::atomic<long> bad{0};
  if (check == "threads") {  // one stage, several threads, fields of several sizes
    HostStage stage;
    StubStream stream;
    const size_t sizes[4] = {8 * 1000, 8 * 40000, 8 * 600000, 8 * 2500000 + 8};
    std::vector<std::thread> ts;
    for (int t = 0; t < 4; ++t)
      ts.emplace_back([&, t] {
        for (int r = 0; r < 12; ++r) bad += read_field(stage, stream, field(sizes[(t + r) % 4], t * 100 + r));
      });
    for (auto& t : ts) t.join();
    reads = 4 * 12;
  }
  std::printf("%ld %ld\n", reads, bad.load());
  return 0;
}
