// attention_capped.hip once more with a gate behind every result (see Q3_GATED in attention_tiles.h). A build of its own, so that calls
// without a gate do not carry its operands: with them in the one build a prompt of 17 rows took 7.9 us and 7.5 without, 64 of 40 rows (32
// heads in groups of four) 32.2 and 28.6.
#define Q3_CAP_GATED 1
#include "attention_capped.hip"
