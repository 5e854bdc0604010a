// dense16_glu.hip — dense16.hip's kernel with gated columns, in a translation unit of its own (compile time).
#include "dense16_impl.h"

void mx_dense16_glu(const void* args, int tile, unsigned n, hipStream_t st) {
    const D16Args& a = *(const D16Args*)args;
#define GO(M_, N_) \
    if (tile == 16 * M_ + N_) dense16_launch<D16_GLU, false, M_, N_>(a, n, st);
    D16_TILES(GO)
#undef GO
}
