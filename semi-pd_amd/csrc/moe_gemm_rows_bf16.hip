// The experts' grouped GEMM in tiles of up to 320 rows (moe_gemm_rows.h) for bf16.  A file for each type, for the compiler's time: it has a body of the K
// loop for every 32 rows, twice.
#include "moe_gemm_rows.h"

namespace semipd {
template int launch_moe_gemm_rows<bf16_t>(bf16_t*, const bf16_t*, const bf16_t*, const G8Group&, int64_t, int, int, int, hipStream_t);
}  // namespace semipd
