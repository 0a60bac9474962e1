// Instances of the tile kernel of the chunked backward: fp32 rows, with the gradient of the uncertainty output.
#include "chunk_bwd_tile.h"

namespace pal {
template int launch_tile_t<float, true>(const BwdArgs&, const TileParts&, hipStream_t);
}
