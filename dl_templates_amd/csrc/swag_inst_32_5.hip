#define DLT_D 32
#define DLT_NCH 5
#include "swag_inst.hpp"
