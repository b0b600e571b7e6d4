// Read-only view of a context's plan for the tests: what the work plan chose
// is not part of the C ABI, but tests of a plan's paths have to know that they
// reach them.
#include "hf_context.h"

extern "C" {

// slots per block of the wave-speed maxima
int probe_ways(const hf_ctx* c) { return c->ways; }

// captured step loops held
int probe_graphs(const hf_ctx* c) { return (int)c->graphs.size(); }

// rows (columns for a transposed item, negated) of each item of a step's main
// launch; returns their number
int probe_items(const hf_ctx* c, int* rows, int max)
{
    for (int i = 0; i < c->main_items && i < max; i++) {
        const int r = c->items[c->main_begin + i].rows;
        rows[i] = r >= 0 ? r : -(-r & 255);
    }
    return c->main_items;
}

}
