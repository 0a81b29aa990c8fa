#define DLT_DK 32
#define DLT_DV 32
#define DLT_FLASH_PART 3
#include "flash_inst.hpp"
