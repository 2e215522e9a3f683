// emu_cells.h -- the per-function deposit and gather over particles listed by
// the box their stencil covers (emu_cells.hip).
#pragma once

#include "emu_internal.h"

namespace emu {

// The three calls: the deposit, the deposit from the fixed scratch (no room
// for records: it lists particles by index), and the gather.
enum class BoxCall { deposit, deposit_static, gather };

// Device scratch of one call on np particles and nk fab cells: the box list,
// the records, the gather's results and combined fields, the scan's storage.
struct BoxScratchSize {
    size_t ints = 0, rec = 0, out = 0, comb = 0, scan = 0, total = 0;
};
BoxScratchSize box_scratch_size(int64_t np, int64_t nk, int nf, BoxCall call);

// List the particles by box, then deposit them into the fab (the caller zeroes
// the deposited components first and folds the ghosts after) or gather the RHS
// of each from it into dst (which may be P itself).  `scratch` holds
// box_scratch_size(...) bytes.  Asynchronous on the context stream.
int box_list_and_run(emu_ctx* ctx, const PView& P, const PView* dst, const Fab& fab, BoxCall call, void* scratch,
                     size_t scratch_bytes);

// The same with the context's scratch, in batches of particles that it holds.
int box_run_batched(emu_ctx* ctx, const PView& P, const PView* dst, const Fab& fab, BoxCall call);

// The context's scratch, grown to `need` bytes (hipMalloc) on first use.
int box_scratch(emu_ctx* ctx, size_t need, void** out);

// The static scratch of the current device: static_scratch_init (at
// emu_create, with the device current) looks up its address once per device;
// static_scratch checks a call's sizes against its capacity and returns it.
int static_scratch_init();
int static_scratch(emu_ctx* ctx, int64_t np, int64_t ncells, void** out, size_t* bytes);

} // namespace emu
