// The sort as fgs_sort_gaussian and fgs_sort_render call it.
#pragma once

#include "tile_rank.h"

namespace fgs {

// What a sort takes, checked without a call of the runtime.
int check_sort(int num_rendered, int width, int height, int block_x, int block_y, const char* list_sorting_space, size_t sorting_size,
               const uint64_t* gaussian_keys_unsorted, const uint32_t* gaussian_values_unsorted,
               const uint64_t* gaussian_keys_sorted, const uint32_t* gaussian_values_sorted, const char* who);

// frame: null, or where the launches of the sort write what the blend needs to know of the tiles (keys without bits above the sorted range, as
// fgs_preprocess makes them); what they did not write is null in it afterwards.  who: the entry point, for the messages.
int sort_impl(int num_rendered, int width, int height, int block_x, int block_y, char* list_sorting_space, size_t sorting_size,
              const uint64_t* gaussian_keys_unsorted, const uint32_t* gaussian_values_unsorted,
              uint64_t* gaussian_keys_sorted, uint32_t* gaussian_values_sorted, FrameTables* frame, void* stream, const char* who);

} // namespace fgs
