#define DLT_D 32
#define DLT_NCH 2
#include "swag_inst.hpp"
