#define DLT_D 32
#define DLT_NCH 6
#include "swag_inst.hpp"
