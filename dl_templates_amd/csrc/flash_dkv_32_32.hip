#define DLT_DK 32
#define DLT_DV 32
#define DLT_FLASH_PART 2
#include "flash_inst.hpp"
