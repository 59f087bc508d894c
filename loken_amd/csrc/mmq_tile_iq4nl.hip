// The f16 tiles of one weight format, experts only (see mmq_tile.h).
#include "mmq_tile.h"

LK_DEFINE_EXPERT_TILES(iq4nl, mmq_tile::TileIq4Nl)
