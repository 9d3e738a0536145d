// The tiled GEMM's plain launches on fp16 weight tiles.
#include "ns2_gemm_tiled.h"

template int ns2tiled::launch_tile<ns2tiled::kF16>(ns2tiled::Tile, const ns2tiled::TGemmArgs&, int);
