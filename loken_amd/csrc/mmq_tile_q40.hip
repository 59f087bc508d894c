// The f16 tiles of one weight format (see mmq_tile.h).
#include "mmq_tile.h"

LK_DEFINE_TILES(q40, mmq_tile::TileQ40)
