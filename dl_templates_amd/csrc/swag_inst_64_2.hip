#define DLT_D 64
#define DLT_NCH 2
#include "swag_inst.hpp"
