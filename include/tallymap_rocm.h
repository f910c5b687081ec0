/* tallymap_rocm.h -- the C ABI of libtallymap_rocm.so, the MI355X (gfx950) launch library of the tallymap_amd
 * kernel backend.  Plain pointers and sizes only.  Every tm_ entry returns 0 on success and a nonzero code on
 * failure; tm_last_error() then holds the message (per thread).  The two tallymap_ entries keep the reference's
 * return conventions.
 *
 * It replaces the reference's CUDA launch shim, tallymap/backends/kernel/shim.cc (and the NVRTC calls of
 * compile.py), entry for entry:
 *   tallymap_register, tallymap_kernel_info: the reference's own names and signatures (shim.cc:134-155), below
 *   tm_register      <- tallymap_register      (shim.cc:134-142), returning an error for an empty image
 *   tm_kernel_info   <- tallymap_kernel_info   (shim.cc:147-155), for any block size and before a launch
 *   tm_launch        <- SjLaunchImpl, the body of the XLA FFI handler TallymapLaunch (shim.cc:157-250), as a
 *                       plain C call: an XLA FFI handler bound for platform "ROCM" forwards its buffers, stream and
 *                       attrs (kernel_id, block, n_zero, flags, n_items) to it
 *   tm_compile       <- compile.compile_cubin's NVRTC sequence (compile.py:160-173), with hipRTC for gfx950
 *   tm_init          <- compile.py's Drv / dlopen of the driver (shim.cc:44-82): binds the HIP runtime the process
 *                       already uses (no second runtime; the library's only device code is the scratch array
 *                       of tm_launch_noalloc, every kernel lives in the program's own code object)
 *   tm_launch_aux    <- _records.canon (_records.py:45-74): the Records canonicalisation, here device passes of the
 *                       program's own module instead of XLA ops
 */
#ifndef TALLYMAP_ROCM_H
#define TALLYMAP_ROCM_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Bind the HIP runtime library `hip_path` and hipRTC library `hiprtc_path` (NULL: the system's libamdhip64.so.7 /
 * libhiprtc.so.7).  Idempotent: later calls with other paths keep the first binding. */
int tm_init(const char* hip_path, const char* hiprtc_path);

/* Compile HIP source `src` with hipRTC (options `opts[0..nopts)`, e.g. --offload-arch=gfx950).  On success
 * *image / *n hold the code object (free with tm_free); *log (may be NULL) receives the compiler log (tm_free). */
int tm_compile(const char* src, const char* name, const char* const* opts, int nopts, void** image, size_t* n,
               char** log);

/* Register code object `image` (n bytes, copied) under `id`.  The first registration of an id wins; `note` is a
 * label for error messages.  Modules are loaded per device lazily, on the first launch there. */
int tm_register(long long id, const void* image, size_t n, const char* note);

/* Launch program `id` on `stream` (a hipStream_t; NULL: the null stream) over n_items items.  bufs: the n buffer
 * pointers in the program's layout ([per-item operands][broadcast operands][results]).  n_zero > 0: run tm_zero
 * first (it clears the program's accumulators and counters); flags bit 1: run tm_post after tm_main (exact
 * readout, truncation poison); flags bit 2 (value 4, spawning programs only, without tm_zero and tm_post): a later
 * generation of a spawn tree, whose item count tm_main reads from the program's control words (written by
 * tm_qnext after the previous generation), n_items its upper bound (the queue capacity), which sizes the grid;
 * flags bit 3 (value 8): run tm_post after tm_main where the launch spread (below), or with n_items 0 (its float64
 * sums of small launches then hold what tm_main left; a launch that did not spread has added to the outputs itself).
 * block: threads per block of tm_main (the program's compiled block size).  The grid is persistent:
 * min(ceil(n_items / block), compute units x blocks per CU), blocks per CU being tm_main's occupancy, or the module's
 * `int tm_grid_cap` (a __constant__, read when the module loads) where that is lower; with `int tm_spread` above 1, a
 * launch of fewer items than those lanes spreads: up to tm_spread lanes per item (idle lanes compute draws ahead).
 * Asynchronous: nothing waits for the kernels. */
int tm_launch(long long id, void* stream, void* const* bufs, int n, int n_zero, int flags, long long n_items,
              int block);

/* Launch the auxiliary entry `name` of program `id` (grid x block threads, the same buffer list and n_items as
 * tm_launch): the passes that move a Records output's raw records to their canonical slots after tm_launch
 * (tm_rscan<j>, tm_rtop<j>, tm_rcanon<j>).  Replaces the reference's canonicalisation after each one-pass launch,
 * done there in XLA ops (_records.py:45-74, canon).  A spawning program's tm_qnext (grid 1, n_items 1 after the
 * roots' launch, else 0) turns a generation's ticket count into the next generation's item count, so the
 * generations of a tree queue back to back without a host read (the reference runs them inside one launch through
 * its ticket ring, backends/kernel/kernel.py:1006-1040).  Asynchronous like tm_launch. */
int tm_launch_aux(long long id, const char* name, void* stream, void* const* bufs, int n, long long n_items,
                  unsigned grid, int block);

/* out[8]: registers per lane of the item loop (tm_main, or tm_adjoint / tm_count / tm_fused in an adjoint), private (scratch) bytes per lane, static LDS bytes per block, achieved
 * blocks per CU at `block` threads, resident threads on the device, compute units, max threads per block, and the
 * grid tm_launch uses for 2^31 - 1 items. */
int tm_kernel_info(long long id, int block, long long out[8]);

const char* tm_last_error(void);
void tm_free(void* p);

/* The reference launch shim's own registry exports, with its signatures and return conventions, so that its
 * compile.py binds this library unchanged (compile.py:215-237):
 *   tallymap_register    <- shim.cc:134-142: copies `n` bytes of the code object `data` under `id`; the first
 *                           registration of an id wins; returns 0 (an empty image registers nothing).
 *   tallymap_kernel_info <- shim.cc:144-155: once the program's item loop has been launched on some device, fills
 *                           out[7] = {registers per lane, private (scratch) bytes per lane, static LDS bytes per
 *                           block, blocks per CU at the launch block size, CUs, max resident threads per CU, block
 *                           size of the first launch} and returns 1; returns 0 before any launch (nothing loaded). */
int tallymap_register(int64_t id, const char* data, size_t n, const char* note);
int tallymap_kernel_info(int64_t id, long long* out);

/* Bytes of the device array tm_launch_noalloc places scratch buffers in (and 16,608 more for the claim counters of a
 * program's item ranges): one per GPU the library runs on, held until the process ends. */
#define TM_NOALLOC_SCRATCH_BYTES (32u << 20)

/* tm_launch for callers that cannot allocate device memory -- code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc.  No counterpart in the reference.  The caller passes the inputs and outputs in
 * bufs as for tm_launch; the n_slots buffers named by slots[] (their bufs entries are ignored and may be NULL) are
 * placed instead, 256-byte aligned and `bytes[j]` long, in the library's own per-device array of
 * TM_NOALLOC_SCRATCH_BYTES: the program's scratch (exact and fixed-point words, the claim / truncation counters,
 * a replay tape).  A layout that does not fit is refused with an error before anything is queued.  tm_zero
 * (n_zero > 0) clears what must start at zero, as for tm_launch; the array otherwise keeps the last call's
 * contents.  Every call on one GPU shares that GPU's array: calls that overlap on one GPU (other streams, other
 * threads) race.  The first call on a device resolves the array there (and loads the program's module, as
 * tm_launch does); later calls allocate nothing. */
int tm_launch_noalloc(long long id, void* stream, void* const* bufs, int n, const int* slots,
                      const long long* bytes, int n_slots, int n_zero, int flags, long long n_items, int block);

#ifdef __cplusplus
}
#endif

#endif
