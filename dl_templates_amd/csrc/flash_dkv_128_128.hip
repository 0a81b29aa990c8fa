#define DLT_DK 128
#define DLT_DV 128
#define DLT_FLASH_PART 2
#include "flash_inst.hpp"
