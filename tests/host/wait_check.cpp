// The wait for a trial's sums on a stand-in for the HIP runtime: it returns when the last
// sum lands, whatever its value; a stream that ends without them, and an error of the
// stream, are reported.
#include "fake_hip.hpp"

#include "sync.hpp"

#include <limits>
#include <vector>

namespace {

std::string refusal(const std::vector<double>& sums, hipStream_t s) {
  try {
    sp::wait_sums(sums.data(), static_cast<int>(sums.size()), s, 50.0);
  } catch (const sp::Error& e) {
    fake::check(e.code == sp::kBackend, "a backend error");
    return e.what();
  }
  return "";
}

}  // namespace

int main() {
  fake::Stream s;
  std::vector<double> sums(7);
  const double inf = std::numeric_limits<double>::infinity();
  const double values[] = {0.0, -0.0, inf, -inf, std::numeric_limits<double>::quiet_NaN(), 1.0, 2.0};
  // Landing one by one, the first last, long after the spin.
  sp::expect_sums(sums.data(), 7);
  fake::stream_status = hipErrorNotReady;
  std::thread device([&] {
    for (int i = 6; i >= 0; --i) {
      std::this_thread::sleep_for(std::chrono::milliseconds(2));
      __atomic_store_n(reinterpret_cast<std::uint64_t*>(&sums[i]),
                       *reinterpret_cast<const std::uint64_t*>(&values[i]), __ATOMIC_RELAXED);
    }
  });
  fake::check(refusal(sums, fake::handle(s)).empty(), "sums that land are awaited");
  fake::check(std::memcmp(sums.data(), values, sizeof values) == 0, "every sum has landed");
  device.join();
  // The stream ends and one sum is missing.
  sp::expect_sums(sums.data(), 7);
  for (int i = 0; i < 6; ++i) sums[i] = values[i];
  fake::stream_status = hipSuccess;
  fake::check(refusal(sums, fake::handle(s)) == "the device ended a trial without its sums",
              "an ended stream without its sums is refused");
  // The stream reports an error.
  fake::stream_status = hipErrorIllegalAddress;
  fake::check(refusal(sums, fake::handle(s)).find("hipError") != std::string::npos ||
                  refusal(sums, fake::handle(s)).find("failed") != std::string::npos,
              "a stream's error is reported");
  std::printf("waits ok\n");
  return 0;
}
