// Switches of the bfloat16 kernel libraries for tests and measurements only: each forces a choice that a
// library otherwise makes by the shape.  They are no part of the product's interface: nothing in the engine
// sets one.  Each of libti_gemm_bf16 and libti_attention_bf16 exports the two functions below; the state is
// the library's (process-wide), and the host library's Ops applies an object's own overrides around its calls
// (Ops::tune) and resets them afterwards.
//
// libti_gemm_bf16:
//   force_tile           1: 256 x 128, 2: 128 x 128; not for SwiGLU 3 / 4: 128 x 64, 6: 64 x 64, 8: 128 x 160, 9: 256 x 160,
//                        11: 256 x 128 by four wavefronts; for SwiGLU alone 5 / 7: 64 x 128, 10 / 12: 256 x 256 (another's number:
//                        128 x 128 for SwiGLU, 128 x 64 for the others); 0: by the shape
//   normed_weight_below  weights of fewer elements keep the norm inside the product (0: the default)
//   normed_groups        1 to 3 groups of four wavefronts, a tile each, in the product with the norm inside (0: by the tiles)
//   tiles_160            0: no tiles of 160 columns
//   tiles_256            0: no tiles of 256 x 256
//   two_ranges           0: never split a product's columns between two tiles
//   xcd_rows             row tiles per block of the order in which a die takes the tiles of a tiled product (-1: the grid's order,
//                        0: by the weight's size)
//   die_order            0: the dies take the tiles of a small weight in the grid's order
//   skinny_waves         4 or 8 wavefronts in the kernel for M <= 64 (0: by the shape)
//   qkv_prep_min_rows    the fewest rows ti_gemm_bf16_qkv_prep serves (17)
//   qkv_prep_rows        64 / 128 / 256: the rows of ti_gemm_bf16_qkv_prep's tile, 512: tiles of 256 x 256; 0: by the shape
//   wide_rows            0: 17..64 rows times a weight of 16,384 rows or more take the other kernels
//   tiled_from           17..64 rows x weight elements from which they take the tiled kernels (280 Mi; 1000 Mi for a product that
//                        stores, K below 4096 and few enough workgroups of 16 rows: set, it holds for both, and rows_112 is off)
//   add_split            0: ti_gemm_bf16_add_split serves nothing
//   use_pipelined        0: the plain tiled kernel for every K
//   row_per_wave         0: few tokens and a weight of few rows take the 16-row kernels too
//   skinny_groups        1 or 2 groups of 16 weight rows a workgroup where 17 to 112 rows come through LDS (0: by the shape)
//   rows_112             0: above 64 rows, and where the weight is large from 17 on, every product takes the tiles
//   rows_staged          0: up to 16 rows never take the kernel whose rows come through LDS stages of each wavefront's own
//   skinny_copy          0: up to 16 tokens, fragments of the token rows straight from memory
//   pieces               0: up to 16 rows never take the kernel with the token rows in pieces
//   skinny_deep          0: four chunks of K in flight per wavefront also for a long K
//   rows_direct          0: the kernel with a weight row per wavefront takes the rows of one and two tokens through LDS too
//   wide_rows_min_n      the fewest weight rows from which 17..64 rows take the kernel that keeps them in registers (16,384)
//   wide_rows_grid       its number of workgroups (0: a tile of 16 weight rows each, at most one per compute unit)
// libti_attention_bf16:
//   prefill_groups       1 or 2 groups of wavefronts per workgroup, 0: by the launch
//   prefill_use_lds      0: the kernel without LDS for every head size
//   decode_stages        1 or 2 LDS stages a wavefront in the decode kernel by records (head size 128), 0: by the launch
#pragma once
#ifdef __cplusplus
extern "C" {
#endif
int ti_tuning_set(const char* name, long value);     // 0, or 1 for a name the library does not know
void ti_tuning_reset();                              // every choice back to the library's own
// libti_gemm_bf16: what is chosen for M rows times N output columns.  The tile (by its number above) and, where the columns are
// split between two (n_big > 0), the second one from column n_big on; the rows of the q/k/v product's tile (0: left to the
// product and the preparation kernel), 256 and 128 where n_big > 0.
int ti_gemm_bf16_tile_choice(int swiglu, int M, int N, int K, int* rest, int* n_big);
int ti_gemm_bf16_qkv_choice(int M, int N, int K, int* n_big);
int ti_gemm_bf16_qkv_wide(int M, int N, int K);      // 1: tiles of 256 x 256 in its place
// ... SwiGLU by quarters (tiles 10 and 12), in place of the first; 0: that one
int ti_gemm_bf16_quarters_ranges(int M, int N, int K, int* rest, int* n_big);
int ti_gemm_bf16_quarters_choice(int M, int N, int K);
// libti_gemm_generic: 1 where float32 rows take the tiles whose wavefronts split their floats together
int ti_gemm_generic_f32_choice(int swiglu, int M, int N, int K, long lda);
#ifdef __cplusplus
}
#endif
