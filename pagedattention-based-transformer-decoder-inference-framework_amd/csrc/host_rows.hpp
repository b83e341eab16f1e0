// Pinned host memory for the rows that steps return (llm_host_rows_take / _give).
#pragma once

#include <cstddef>

namespace llm {

// An engine whose decode steps return `bytes` at most begins, or the last one ends: what is
// free is given back then.
void host_rows_engine_begins(size_t bytes);
void host_rows_engine_ends();

}  // namespace llm
