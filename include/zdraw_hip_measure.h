/*
 * zdraw_hip_measure.h: measurement aids of libzdraw_hip.so. NOT FOR CALLERS.
 *
 * Nothing here has a counterpart in the reference's bridge (src/metal/metal_c.zig) and a
 * renderer never calls any of it: the benchmark and the tests use these entries to choose
 * between builds of one kernel and to read the shader clock a launch really ran at. They
 * change process-wide state and are not part of the drop-in boundary (include/zdraw_hip.h).
 *
 * The library itself reads no environment variable for any of this.
 */
#ifndef ZDRAW_HIP_MEASURE_H
#define ZDRAW_HIP_MEASURE_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Clock probe. While on, every workgroup of an attention launch records how long it ran in
 * shader-clock cycles and in ticks of the fixed 100 MHz reference counter; cycles / ticks x
 * 0.1 is the clock in GHz that the kernel really ran at (under load the power limit sets
 * it). clock_probe_read waits for the last probed launch and copies the first `capacity`
 * workgroups' figures (in launch order); it returns how many. */
void zdraw_hip_clock_probe(int on);
size_t zdraw_hip_clock_probe_read(uint64_t* cycles, uint64_t* ref_ticks, size_t capacity);

/* Which build of the attention kernel runs. Bit 0: 0 = 8 waves x 32 query rows per
 * workgroup, one workgroup per CU (default); 1 = 4 waves x 32 query rows, two workgroups
 * per CU. Bit 1: 2 = never split the tiles of a thinly filled last round along the keys
 * (by default they are). Bit 2: 4 = 256-row tiles also where a small launch would take
 * 128-row tiles with two key groups. */
void zdraw_hip_set_attention_variant(int variant);

/* The tiles that a launch of prepared (or bf16) operands takes by default on a device with `cus`
 * compute units: `heads` = segments x heads, `keys` = tokens or the key limit. *rows = query rows per
 * tile (256, or 128 with two key groups); *tail_tiles and *splits as zdraw_hip_attention_tail_plan
 * gives them. Host arithmetic only. */
void zdraw_hip_attention_plan(uint64_t heads, uint32_t tokens, uint32_t keys, uint32_t cus, uint32_t* rows, uint32_t* tail_tiles,
                              uint32_t* splits);

/* Which build multiplies 256 x 256 tiles of 16-bit activations. 1 = four waves, 128 x 128
 * each (default); 0 = eight waves, 64 x 128 each. 2 = every product on the kernel that
 * addresses A and W through pointers and takes no scratch. */
void zdraw_hip_set_gemm_build(int build);

/* The tile of C (rows x columns) that `groups` (1..3) side-by-side products C[m][n] =
 * A[m][k] x W[n][k]^T run on, on a device with `cus` compute units. Host arithmetic only. */
void zdraw_hip_gemm_tile(uint32_t m, uint32_t k, uint32_t n, uint32_t groups, uint32_t cus, uint32_t* rows, uint32_t* cols);

/* How many of `rows` rows of a 16-bit A or W (`ld` elements apart, k of them used) one launch of a
 * product takes: all, unless they span all but 4 GiB; 0 where not even one row fits the kernels'
 * 32-bit offsets. A product is cut accordingly. Host arithmetic only. */
void zdraw_hip_gemm_launch_rows(uint32_t rows, uint64_t ld, uint32_t k, uint32_t* per_launch);

/* Key ranges per query tile of a wide head of `tokens` tokens on a device with `cus` compute units,
 * and the bytes of scratch that their shares take. Host arithmetic only. */
void zdraw_hip_wide_ranges(uint32_t tokens, uint32_t cus, uint32_t* ranges, uint64_t* share_bytes);

/* From here on a scratch slot may not grow past `bytes`: what a call does when the device has no
 * more memory. 0 = no limit (default). */
void zdraw_hip_set_scratch_limit(size_t bytes);

/* How many query tiles (128 rows) of the last wide-head launch had a score outgrow its row's
 * fixed reference point and were formed again with a running maximum (waits for that
 * launch). 0 on ordinary data; -1 if no wide-head launch has been made or the read failed. */
int zdraw_hip_wide_redo_tiles(void);

/* A queue as zdraw_hip_create_queue makes it, its stream confined to cu_count compute units
 * (0 < cu_count < the device's CU count; anything else: an ordinary queue): does a kernel's
 * time follow the CU count or the board's power limit. */
void* zdraw_hip_create_queue_on_cus(void* device, int cu_count);

#ifdef __cplusplus
}
#endif
#endif
