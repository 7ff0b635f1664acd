// tensor.hip with the storage of its kernels' dynamic LDS (and the attribute's
// spelling that may follow a storage class)
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#define alignas(n) __attribute__((aligned(n)))
#include "../../eom-imsrg_full_amd/csrc/tensor.hip"
namespace {
thread_local double rows[20480];
}
