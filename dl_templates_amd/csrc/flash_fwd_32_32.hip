#define DLT_DK 32
#define DLT_DV 32
#define DLT_FLASH_PART 0
#include "flash_inst.hpp"
