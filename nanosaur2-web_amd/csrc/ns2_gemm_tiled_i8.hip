// The tiled GEMM's plain launches on int8 weight tiles.
#include "ns2_gemm_tiled.h"

template int ns2tiled::launch_tile<ns2tiled::kI8>(ns2tiled::Tile, const ns2tiled::TGemmArgs&, int);
