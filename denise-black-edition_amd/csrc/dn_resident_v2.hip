// Chip-resident time loop, FDORDER 4, viscoelastic P/SV.
#define DN_F 2
#define DN_GROUP 2
#include "dn_resident_inst.inc"
