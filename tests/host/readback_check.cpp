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
// one read of field f, slot by slot or by a plain copy; the bytes that differ
static std::atomic<long> rings{0};
static long read_field(ReadPool& pool, StubStream& stream, const std::vector<char>& f, double gain) {
  std::vector<char> out(f.size());
  const hipError_t e = read_back(
      pool, &stream, out.data(), f.size(), gain,
      [&](char* pin, size_t off, size_t len) {
        rings += off == 0;
        std::memcpy(pin, f.data() + off, len);
        std::this_thread::yield();
        return hipSuccess;
      },
      [&] {
        std::memcpy(out.data(), f.data(), f.size());
        return hipSuccess;
      });
  if (e != hipSuccess) return (long)f.size();
  long bad = 0;
  for (size_t i = 0; i < f.size(); ++i) bad += out[i] != f[i];
  return bad;
}
static long expect(bool ok, const char* what) {
  if (!ok) std::fprintf(stderr, "%s\n", what);
  return !ok;
}

int main(int argc, char** argv) {
  const std::string check = argc > 1 ? argv[1] : "";
  long reads = 0;
  std::atomic<long> bad{0};
  StubStream stream;
  ReadPool pool;
  if (check == "threads") {  // several threads, fields of several sizes
    pool.owed = 1e9;  // pinned whenever a ring is free
    ReadPoolUser user(pool);
    const size_t sizes[4] = {8 * 1000, 8 * 40000, 8 * 600000, 8 * 2500000 + 8};
    std::vector<std::thread> ts;
    for (int t = 0; t < 4; ++t)
      ts.emplace_back([&, t] {
        for (int r = 0; r < 12; ++r) bad += read_field(pool, stream, field(sizes[(t + r) % 4], t * 100 + r), 100.);
      });
    for (auto& t : ts) t.join();
    reads = 4 * 12;
    bad += expect(rings > 4, "the rings were hardly used");
    bad += expect(stub_pinned <= 2 * (16l << 20), "more than two rings of 16 MB");
  } else if (check == "pinning") {  // what a first read and a later one pin
    const size_t small = 8 * 1000, mid = 8 * 131072, big = 57u << 20;  // 8 KB, 1 MB, 57 MB
    {
      ReadPoolUser a(pool), b(pool);
      bad += read_field(pool, stream, field(mid, 1), array_gain(mid));
      bad += read_field(pool, stream, field(small, 2), formed_gain(small));
      bad += expect(stub_pins == 0, "one read of a case pins memory that costs more than it gains");
      for (int r = 0; r < 50; ++r) bad += read_field(pool, stream, field(small, r), array_gain(small));
      bad += expect(stub_pins == 0, "a small array is read by a plain copy");
      for (int r = 0; r < 3; ++r) bad += read_field(pool, stream, field(small, r), formed_gain(small));
      bad += expect(stub_pins == 1 && stub_pinned <= (64l << 10), "several small formed reads pin one small ring");
      for (int r = 0; r < 9; ++r) bad += read_field(pool, stream, field(mid, r), array_gain(mid));
      bad += expect(stub_pins == 2 && stub_pinned <= (1l << 20), "several reads of 1 MB pin as much");
      bad += read_field(pool, stream, field(big, 3), array_gain(big));
      bad += expect(stub_pins == 3 && stub_pinned <= (16l << 20), "a large read pins one ring of 16 MB");
    }
    bad += expect(stub_pinned == 0, "pinned memory is given back with the last case");
    {
      ReadPoolUser c(pool);
      const long pins = stub_pins;
      bad += read_field(pool, stream, field(mid, 5), array_gain(mid));
      bad += expect(stub_pins == pins, "the next case starts without pinned memory");
    }
    reads = 66;
  }
  if (check == "short") {  // no pinned memory to be had, then some
    pool.owed = 1e9;
    ReadPoolUser user(pool);
    const size_t sizes[3] = {8 * 1000, 8 * 600000, 8 * 2500000 + 8};
    for (size_t most : {(size_t)0, (size_t)(20u << 10), (size_t)(1u << 20)}) {
      stub_most = most;
      for (size_t n : sizes) bad += read_field(pool, stream, field(n, (unsigned)n), 100.);
      bad += expect(stub_pinned <= (long)most, "more than can be pinned");
    }
    for (HostStage& r : pool.ring) bad += expect(!r.busy, "a ring was not given back");
    reads = 9;
  }
  if (check == "device") {  // a case of device 1, read by a thread whose current device is 0
    pool.owed = 1e9;
    ReadPoolUser user(pool);
    StubStream other{1};
    for (size_t n : {(size_t)8 * 1000, (size_t)8 * 600000}) {
      bad += read_field(pool, other, field(n, 7), 100.);
      bad += read_field(pool, stream, field(n, 8), 100.);
    }
    bad += expect(rings == 4, "the rings were not used");
    bad += expect(stub_device == 0, "the thread's device was changed");
    reads = 4;
  }
  std::printf("%ld %ld\n", reads, bad.load());
  return 0;
}
