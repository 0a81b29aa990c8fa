#define DLT_D 64
#define DLT_NCH 3
#include "swag_inst.hpp"
