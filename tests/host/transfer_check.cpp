// The pipelined copies of large fields on a stand-in for the HIP runtime: every size comes
// back bit for bit, the pinned slots are made when they pay and freed, and a refusal of
// pinned memory leaves plain copies.
#include "fake_hip.hpp"

#include "transfer.cpp"

#include <vector>

namespace {

constexpr std::size_t MB = 1UL << 20;

void fill(std::vector<unsigned char>& v, unsigned seed) {
  for (std::size_t i = 0; i < v.size(); ++i)
    v[i] = static_cast<unsigned char>((seed = seed * 1664525u + 1013904223u) >> 24);
}

// `host` to the device and back through `t`.
void round_trip(sp::Transfer& t, fake::Stream& s, std::size_t bytes, unsigned seed) {
  std::vector<unsigned char> host(bytes), device(bytes), back(bytes);
  fill(host, seed);
  t.upload(device.data(), host.data(), bytes, fake::handle(s));
  fake::check(device == host, "an upload");
  t.download(back.data(), device.data(), bytes, fake::handle(s));
  fake::check(back == host, "a download");
}

}  // namespace

int main() {
  fake::Stream s;
  {
    // Loaded and read once, a field below 32 MB makes no slots; nor do small ones ever.
    sp::Transfer t;
    round_trip(t, s, 8 * MB, 1);
    round_trip(t, s, 32 * MB - 16, 2);
    fake::check(fake::pinned_allocations == 0, "no slots for a first field below 32 MB");
    for (unsigned k = 0; k < 12; ++k) round_trip(t, s, 8 * MB - 16, 3 + k);
    fake::check(fake::pinned_allocations == 0, "no slots for fields below 8 MB");
  }
  {
    // Read again and again, it does, once.
    sp::Transfer t;
    for (unsigned k = 0; k < 10; ++k) round_trip(t, s, 8 * MB + 1000, k);
    fake::check(fake::pinned_allocations == 1, "slots after 64 MB of plain copies");
    const int before = fake::copies;
    round_trip(t, s, 8 * MB + 1000, 99);
    fake::check(fake::copies - before == 1 + 9, "a plain upload and nine chunks back");
    // Every size through the slots: whole chunks, remainders, more than the lanes' slots.
    for (std::size_t bytes : {8 * MB, 8 * MB + 16, 11 * MB - 48, 31 * MB, 32 * MB, 33 * MB + 80})
      round_trip(t, s, bytes, static_cast<unsigned>(bytes));
    fake::check(fake::pinned_allocations == 1, "the slots are kept");
  }
  fake::check(fake::pinned_alive == 0, "the slots are freed");
  {
    // A field of 32 MB makes them at once, in its download; its upload does not.
    sp::Transfer t;
    std::vector<unsigned char> host(32 * MB), device(32 * MB);
    t.upload(device.data(), host.data(), host.size(), fake::handle(s));
    fake::check(fake::pinned_allocations == 1, "an upload makes no slots");
    round_trip(t, s, 32 * MB, 7);
    fake::check(fake::pinned_allocations == 2, "a download of 32 MB makes them");
  }
  {
    // Pinned memory refused: plain copies, and no second attempt.
    sp::Transfer t;
    fake::refuse_pinned = true;
    round_trip(t, s, 40 * MB + 16, 11);
    fake::refuse_pinned = false;
    const int before = fake::copies;
    round_trip(t, s, 70 * MB, 12);
    fake::check(fake::copies - before == 2, "plain copies after a refusal");
    fake::check(fake::pinned_alive == 0, "nothing pinned after a refusal");
  }
  std::printf("transfers ok\n");
  return 0;
}
