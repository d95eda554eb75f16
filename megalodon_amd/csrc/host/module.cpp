// The extension module megalodon_amd._host.
#include "host.hpp"

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  mega_host::bind_decode(m);
  mega_host::bind_ops(m);
}
