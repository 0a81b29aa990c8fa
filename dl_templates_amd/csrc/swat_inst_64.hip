#define DLT_D 64
#include "swat_inst.hpp"
