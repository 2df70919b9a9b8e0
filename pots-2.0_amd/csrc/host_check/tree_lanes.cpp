// The outer Merkle tree's kernel on the CPU, lane by lane (lanes/hip/hip_runtime.h):
//
//   tree_lanes N [last-first] < N 32-byte digests > the 2N - 1 nodes in pre-order
#include "../merkle.hip"

namespace pots {

void note_hip_error(hipError_t, const char*, const char*, int) {}
void note_error(const std::string&) {}
int arena_get(int, size_t, void**) { return POTS_E_NOMEM; }
bool is_device_pointer(const void*) { return true; }

}  // namespace pots

int main(int argc, char** argv) {
  const size_t n = argc > 1 ? strtoull(argv[1], nullptr, 10) : 0;
  if (n == 0) return 1;
  lanes::g_last_first = argc > 2;
  std::vector<uint4> leaves(2 * n), nodes(2 * (2 * n - 1));
  if (fread(leaves.data(), 32, n, stdin) != n) return 1;
  if (pots_merkle_tree_async(n, reinterpret_cast<const uint8_t*>(leaves.data()),
                             reinterpret_cast<uint8_t*>(nodes.data()), nullptr) != POTS_E_OK)
    return 1;
  return fwrite(nodes.data(), 32, 2 * n - 1, stdout) == 2 * n - 1 ? 0 : 1;
}
