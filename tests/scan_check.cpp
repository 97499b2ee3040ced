// The pre-pass's verdict on a meshlet that ends early (scan_meshlet,
// stride_lane.h), on the host: a meshlet of one strip whose bit range is cut
// after every bit, with the strip length given.
//
//   scan_check <strip length>
//
// Prints the error code (MeshletScan::error) for every cut, 1 bit to all.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../meshpress_amd/csrc/stride_lane.h"

using namespace stride;

int main(int argc, char** argv) {
  if (argc < 2) return 1;
  // header (3 locals, 1 triangle, 1 strip), the strip length, three raw ids of
  // 2 bits, three 8-bit anchors, six coders Rice(0), two deltas of 0 an axis
  std::vector<int> bits;
  auto put = [&](uint32_t v, int n) {
    while (n--) bits.push_back((v >> n) & 1u);
  };
  for (uint32_t v : {3u, 1u, 1u, (uint32_t)std::atoi(argv[1])}) put(v, 16);
  for (uint32_t v = 0; v < 3; ++v) put(4u | v, 3);
  for (int d = 0; d < 3; ++d) put(77, 8);
  for (int j = 0; j < 6; ++j) put(0x100, 16);
  for (int j = 0; j < 6; ++j) put(1, 1);
  std::vector<uint32_t> words((bits.size() + 31) / 32 + 4, 0);
  for (size_t i = 0; i < bits.size(); ++i)
    if (bits[i]) words[i >> 5] |= 1u << (8 * ((i & 31) >> 3) + 7 - (i & 7));
  const int32_t g_bits[3] = {8, 8, 8};
  for (uint32_t end = 1; end <= bits.size(); ++end) {
    MeshletScan s;
    scan_meshlet(GlobalWords{words.data(), (end + 31u) / 32u + 2u}, 0, end, g_bits, s);
    std::printf("%u\n", s.error);
  }
  return 0;
}
