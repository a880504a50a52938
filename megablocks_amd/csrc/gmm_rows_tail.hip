// NN / NT products of 16-bit operands, k a multiple of 8 but not of the K tile: see KTAIL in gmm_dma.h.
#include "gmm_rows.h"

namespace mbx {

int gmm_rows_tail(const DmaCall& call) { return dispatch_rows<true>(call); }

#ifdef MBX_TICKS
int gmm_rows_tail_set_ticks(void* buffer) { return (int)hipMemcpyToSymbol(HIP_SYMBOL(dma::g_ticks), &buffer, sizeof(buffer)); }
#endif

}  // namespace mbx
