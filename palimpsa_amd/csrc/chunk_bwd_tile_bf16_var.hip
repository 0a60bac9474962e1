// Instances of the tile kernel of the chunked backward: bf16 rows, with the gradient of the uncertainty output.
#include "chunk_bwd_tile.h"

namespace pal {
template int launch_tile_t<bf16_t, true>(const BwdArgs&, const TileParts&, hipStream_t);
}
