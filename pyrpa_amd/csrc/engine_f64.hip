#include "engine_impl.h"

namespace gmod {
template class ConvEngine<double>;
}  // namespace gmod
