#define DLT_D 32
#define DLT_NCH 3
#include "swag_inst.hpp"
