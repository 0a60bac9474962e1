// Instances of the tile kernel of the chunked backward: bf16 rows, without the gradient of the uncertainty output.
#include "chunk_bwd_tile.h"

namespace pal {
template int launch_tile_t<bf16_t, false>(const BwdArgs&, const TileParts&, hipStream_t);
}
