#define DLT_D 64
#define DLT_NCH 4
#include "swag_inst.hpp"
