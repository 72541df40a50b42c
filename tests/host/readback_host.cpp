// csrc/readback.hpp on the host, over the runtime calls of hip/hip_runtime.h.
// readback_host CASE
#include <chrono>
#include <condition_variable>
#include <functional>
#include <string>

#include "../../gpucelllistsph.jl_amd/csrc/readback.hpp"

using namespace gclsph;

namespace {
int failures = 0;
void expect(bool ok, const char* what) {
  if (!ok) std::printf("%s\n", what), ++failures;
}

// out from src by a stream that writes at once
void copy(std::vector<char>& out, const std::vector<char>& src, hipStream_t st) {
  HostSlots::copy_out(out.data(), out.size(), st, [&](void* slot, size_t off, size_t len) {
    std::memcpy(slot, src.data() + off, len);
  });
}
std::vector<char> pattern(size_t bytes, unsigned seed) {
  std::vector<char> v(bytes);
  for (size_t i = 0; i < bytes; ++i) v[i] = char((i * 31 + (i >> 12) + seed) & 0x7f);
  return v;
}

// A copy waits for its own stream only: the first one's stream ends when the
// second one's copy is done.
void overlap(size_t bytes) {
  HostSlots::Ref a, b;
  std::mutex m;
  std::condition_variable cv;
  bool second_done = false, first_waits = false, late = false;
  ihipStream_t slow, quick;
  slow.wait = [&] {
    std::unique_lock<std::mutex> l(m);
    first_waits = true;
    cv.notify_all();
    if (!cv.wait_for(l, std::chrono::seconds(20), [&] { return second_done; })) late = true;
  };
  const auto src = pattern(bytes, 1), src2 = pattern(bytes, 2);
  std::vector<char> out(bytes), out2(bytes);
  std::thread first([&] { copy(out, src, &slow); });
  std::thread second([&] {
    {
      std::unique_lock<std::mutex> l(m);
      cv.wait(l, [&] { return first_waits; });
    }
    copy(out2, src2, &quick);
    std::lock_guard<std::mutex> l(m);
    second_done = true;
    cv.notify_all();
  });
  first.join();
  second.join();
  expect(!late, "a copy waited for another stream's work");
  expect(out == src && out2 == src2, "wrong bytes");
}

// Many copies at once; the page-locked memory kept afterwards is bounded, and
// given back with the last object.
void many() {
  {
    HostSlots::Ref a;
    std::vector<std::thread> pool;
    std::mutex m;
    for (unsigned t = 0; t < 24; ++t)
      pool.emplace_back([&, t] {
        ihipStream_t st;
        for (size_t bytes : {size_t(1), HostSlots::kSlot, HostSlots::kSlot + 1, 11 * HostSlots::kSlot - 3}) {
          const auto src = pattern(bytes, t);
          std::vector<char> out(bytes);
          copy(out, src, &st);
          std::lock_guard<std::mutex> l(m);
          expect(out == src, "wrong bytes");
        }
      });
    for (auto& t : pool) t.join();
    expect(pinned_bytes() <= int64_t(HostSlots::kKept * HostSlots::kSlots * HostSlots::kSlot), "too much is kept");
  }
  expect(pinned_bytes() == 0, "page-locked memory is left");
}

// The caller learns what failed: a launch, or the work of the stream.
void errors() {
  HostSlots::Ref a;
  for (size_t chunks : {1, 2, 3, 20}) {
    for (size_t bad : {size_t(0), chunks / 2, chunks - 1}) {
      std::vector<char> out(chunks * HostSlots::kSlot);
      ihipStream_t st;
      std::string got;
      try {
        HostSlots::copy_out(out.data(), out.size(), &st, [&](void*, size_t off, size_t) {
          if (off == bad * HostSlots::kSlot) throw Error(kErrHip, "launch: out of resources");
        });
      } catch (const Error& e) {
        if (e.code == kErrHip) got = e.what();
      }
      expect(got == "launch: out of resources", "a failed launch is reported otherwise");
    }
    std::vector<char> out(chunks * HostSlots::kSlot);
    ihipStream_t st;
    st.result = hipErrorUnknown;
    std::string got;
    try {
      copy(out, out, &st);
    } catch (const Error& e) {
      if (e.code == kErrHip) got = e.what();
    }
    expect(got.find("unknown error") != std::string::npos, "a failed stream is reported otherwise");
  }
}

// A thread whose current device is not the stream's reads as any other, and keeps
// its device.
void devices() {
  HostSlots::Ref a;
  for (int current : {0, 1}) {
    for (size_t bytes : {size_t(1000), 9 * HostSlots::kSlot + 5}) {
      current_device = current;
      ihipStream_t st;
      st.device = 1;
      const auto src = pattern(bytes, 3);
      std::vector<char> out(bytes);
      std::atomic<int> elsewhere{0};
      try {
        HostSlots::copy_out(out.data(), bytes, &st, [&](void* slot, size_t off, size_t len) {
          elsewhere += current_device != st.device;
          std::memcpy(slot, src.data() + off, len);
        });
      } catch (const Error& e) {
        expect(false, e.what());
      }
      expect(out == src, "wrong bytes");
      expect(elsewhere == 0, "a launch with another device current");
      expect(current_device == current, "the thread's device changed");
    }
  }
}
}  // namespace

int main(int, char** argv) {
  const std::string what = argv[1];
  if (what == "overlap") {
    overlap(1000);
    overlap(9 * HostSlots::kSlot + 5);
  } else if (what == "many") {
    many();
  } else if (what == "errors") {
    errors();
  } else if (what == "devices") {
    devices();
  }
  return failures ? 1 : 0;
}
