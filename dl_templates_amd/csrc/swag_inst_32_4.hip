#define DLT_D 32
#define DLT_NCH 4
#include "swag_inst.hpp"
