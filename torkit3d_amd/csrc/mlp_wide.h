// The wide products of mlp_wide.hip, for the entry points of mlp.hip. Slots and splits are 0 where the sizes
// are those of another kernel.
#pragma once

#include "tk3d_common.h"
#include "tk3d_mlp.h"

int tk_mlp_wide_outer_splits(const tk3d_mlp_outer &p);
int tk_mlp_wide_outer(int row, int col, const tk3d_mlp_outer &p, hipStream_t stream);
int tk_mlp_wide_product_slots(int in, int out, const tk3d_mlp_product &p);
int tk_mlp_wide_product(int in, int out, const tk3d_mlp_product &p, hipStream_t stream);
