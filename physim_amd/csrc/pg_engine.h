// Internal declarations shared by the engine's translation units.
#pragma once

#include "physim_gpu.h"

// Records a formatted error message for pg_last_error() and returns `code`.
int pg_set_error(int code, const char* fmt, ...);

// What simulations stepped together (one kind and precision) ask of the batch
// scratch.
struct pg_group_need {
    int32_t kind = PG_KIND_DIRECT, precision = PG_PREC_MIXED;
    uint64_t bodies = 0;
    uint32_t segs = 0, blocks = 0;
    uint64_t lines = 0, most = 0;  // direct sum: lines of partial sums, of a target tile at most
};
void pg_group_add(pg_group_need* g, uint64_t n);
// Device memory the engine holds with one more simulation of `n` bodies, once
// each of the groups has been stepped.
uint64_t pg_engine_bytes_with(pg_engine* e, const pg_group_need* groups, size_t count, uint64_t n);

// The plugin's engine (created on first use, PHYSIM_GPU_DEVICE selects the
// device) and the device transform of one of its gravity elements: false
// when `element` is not a live GPU gravity element of this library.
pg_engine* pg_plugin_engine(void);
bool pg_plugin_element_params(const void* element, pg_params* out);
