// NN / NT products of 16-bit operands, k a multiple of the K tile (64).
#include "gmm_rows.h"

namespace mbx {

int gmm_rows(const DmaCall& call) { return dispatch_rows<false>(call); }

#ifdef MBX_TICKS
int gmm_rows_set_ticks(void* buffer) { return (int)hipMemcpyToSymbol(HIP_SYMBOL(dma::g_ticks), &buffer, sizeof(buffer)); }
#endif

}  // namespace mbx
