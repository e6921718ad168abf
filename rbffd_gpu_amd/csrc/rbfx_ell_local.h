// Device build of an operator set's tile tables (rbfx_ell_build_local).
#pragma once
#include "rbfx_ell_common.h"

struct LocalTables {
    int32_t* pos = nullptr;    // n_tiles + 1 first positions
    int32_t* off = nullptr;    // n_tiles + 1 list offsets
    int32_t* nodes = nullptr;  // the tiles' node lists, ascending
    uint16_t* idx = nullptr;   // every layout entry's place in its tile's list
    int n_tiles = 0, k_max = 0;
};

// Builds the tables of rbfx_build_local_tables for e's layout on its context's stream (complete
// on return). Returns false, with nothing allocated, when the stencils are too wide or a tile's
// list too long for the kernels' LDS tables (the host build serves those); otherwise *rc holds
// the status.
bool rbfx_local_tables_device(rbfx_ell* e, int lt, int cap, size_t lds_limit, LocalTables* T, int* rc);
