#define DLT_DK 64
#define DLT_DV 64
#define DLT_FLASH_PART 3
#include "flash_inst.hpp"
