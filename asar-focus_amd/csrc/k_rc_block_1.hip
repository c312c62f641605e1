#define ASARF_RC_BLOCK_UNIT 1
#include "k_rc_block.hip"
