// Checks of HostTransfers (fx_hostcopy.hpp) against the HIP calls of hip/hip_runtime.h beside this
// file; the check to run is the argument.
#include <cstdio>
#include <string>
#include <vector>

#include "fx_hostcopy.hpp"

using fx::HostTransfers;

namespace {

constexpr size_t MIB = (size_t)1 << 20;

#define REQUIRE(x)                                                            \
  do {                                                                        \
    if (!(x)) {                                                               \
      std::printf("line %d: %s\n", __LINE__, #x);                             \
      return 1;                                                               \
    }                                                                         \
  } while (0)

// up and down through a context's transfers: the bytes come back
bool round_trip(HostTransfers &t, fakeStream &st, size_t bytes)
{
  std::vector<char> a(bytes), dev(bytes), b(bytes);
  for (size_t i = 0; i < bytes; i += 511) a[i] = (char)(i * 2654435761u >> 7);
  return t.copy(dev.data(), a.data(), bytes, hipMemcpyHostToDevice, &st) == hipSuccess &&
         t.copy(b.data(), dev.data(), bytes, hipMemcpyDeviceToHost, &st) == hipSuccess && a == b;
}

// a context's transfers while its device is not the calling thread's current one
int other_device()
{
  for (int current : {0, 1, 2}) {
    fake::current = current;
    for (int device : {0, 1}) {
      HostTransfers t;
      t.device = device;
      fakeStream st{device};
      for (int r = 0; r < 2; r++) REQUIRE(round_trip(t, st, 80 * MIB + 12345));
      REQUIRE(fake::current == current);
    }
  }
  REQUIRE(fake::staged > 0 && fake::pinned == 0);
  return 0;
}

// contexts of one upload and one download each have no workers made; those of a busier context
// serve all of the device and go with the last that used them
int workers_where_they_repay()
{
  fakeStream st{0};
  for (int request = 0; request < 3; request++) {
    HostTransfers t;
    t.device = 0;
    REQUIRE(round_trip(t, st, 20 * MIB));
  }
  REQUIRE(fake::mallocs == 0 && fake::staged == 0);
  HostTransfers *a = new HostTransfers, *b = new HostTransfers;
  a->device = b->device = 0;
  for (int r = 0; r < 4; r++) REQUIRE(round_trip(*a, st, 20 * MIB));
  REQUIRE(fake::pinned > 0 && fake::staged > 0);
  const int chunks = fake::mallocs, staged = fake::staged;
  REQUIRE(round_trip(*b, st, 20 * MIB));
  REQUIRE(fake::mallocs == chunks && fake::staged > staged);
  delete a;
  REQUIRE(fake::pinned == chunks);
  REQUIRE(round_trip(*b, st, 20 * MIB));
  delete b;
  REQUIRE(fake::pinned == 0);
  return 0;
}

// the sizes at which the staged copy takes over, for each direction
int sizes()
{
  fakeStream st{0};
  HostTransfers t;
  t.device = 0;
  for (int r = 0; r < 2; r++) REQUIRE(round_trip(t, st, 40 * MIB));
  std::vector<char> a(16 * MIB), b(16 * MIB);
  auto staged = [&](hipMemcpyKind kind, size_t bytes) {
    const int before = fake::staged, plain = fake::plain;
    if (t.copy(b.data(), a.data(), bytes, kind, &st) != hipSuccess) return -1;
    return (fake::staged > before) != (fake::plain > plain) ? (int)(fake::staged > before) : -1;
  };
  REQUIRE(staged(hipMemcpyHostToDevice, 9 * MIB - 1) == 0 && staged(hipMemcpyHostToDevice, 9 * MIB) == 1);
  REQUIRE(staged(hipMemcpyDeviceToHost, 5 * MIB - 1) == 0 && staged(hipMemcpyDeviceToHost, 5 * MIB) == 1);
  return 0;
}

// without memory for the chunks: plain copies, and one attempt a context
int no_memory()
{
  fakeStream st{0};
  fake::no_memory = true;
  HostTransfers t;
  t.device = 0;
  for (int r = 0; r < 4; r++) REQUIRE(round_trip(t, st, 70 * MIB));
  REQUIRE(fake::mallocs == 1 && fake::staged == 0 && fake::plain == 8);
  fake::no_memory = false;
  HostTransfers u;
  u.device = 0;
  REQUIRE(round_trip(u, st, 70 * MIB) && fake::staged > 0);
  const int plain = fake::plain;
  REQUIRE(round_trip(t, st, 70 * MIB) && fake::plain == plain);  // another context's workers
  return 0;
}

}  // namespace

int main(int, char **argv)
{
  const std::string check = argv[1];
  if (check == "other_device") return other_device();
  if (check == "workers_where_they_repay") return workers_where_they_repay();
  if (check == "sizes") return sizes();
  if (check == "no_memory") return no_memory();
  std::printf("no check %s\n", argv[1]);
  return 2;
}
