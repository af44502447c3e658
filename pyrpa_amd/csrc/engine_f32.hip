#include "engine_impl.h"

namespace gmod {
extern template class ConvEngine<double>;
template class ConvEngine<float>;
}  // namespace gmod
