#define ASARF_RC_BLOCK_UNIT 2
#include "k_rc_block.hip"
