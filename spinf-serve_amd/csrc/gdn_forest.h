// Shared by the plan compiler (gdnplan.cpp) and the forest kernel (gdn_forest.hip).
#pragma once
#define GDN_FOREST_BLOCK 32   // tokens per block
#define GDN_FOREST_DEPTH 64   // tokens on a path inside a forest, at most (rows of the kernel's stack)
// A block's entry in the table, int32: [32] tensor rows (-1: none); [32] bit masks of the tokens above in the block; [32] packed bytes:
// how many rows of the block's path (the tokens above its first token, in earlier blocks) are above the token; 1 + depth of a token that
// is on the next block's path (else 0); and, alike in all 32, the length of this block's path and of the next one's.
#define GDN_FOREST_INTS 96
