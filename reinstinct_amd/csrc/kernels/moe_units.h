// Work of a workgroup column of moe_wide.h, as rein_moe_list_units (moe_expert_sort.hip) writes it
#pragma once

#include "rein_common.h"

struct ReinMoeUnit { unsigned expert, tile, tok, n; };                   // first tile, first sorted entry, entries
