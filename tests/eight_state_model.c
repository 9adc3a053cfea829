/*
   A made-up excitable membrane of 8 states in the form the code generator reads: the
   largest model that takes the chunked kernels, with as many exponentials as states
   allow (two per gate), for the tests of generated models.

   There are a total of 17 entries in the algebraic variable array.
   There are a total of 8 entries in each of the rate and state variable arrays.
   There are a total of 4 entries in the constant variable array.
 */
void
initConsts(double* CONSTANTS, double* RATES, double *STATES)
{
STATES[0] = -70.0;
STATES[1] = 0.02;
STATES[2] = 0.9;
STATES[3] = 0.1;
STATES[4] = 0.1;
STATES[5] = 0.2;
STATES[6] = 0.3;
STATES[7] = 0.4;
CONSTANTS[0] = 0;
CONSTANTS[1] = 90.0;
CONSTANTS[2] = 25.0;
CONSTANTS[3] = 0.4;
}
void
computeRates(double VOI, double* CONSTANTS, double* RATES, double* STATES, double* ALGEBRAIC)
{
ALGEBRAIC[0] = 3.0/(1.0+exp(-(STATES[0]+32.0)/9.0));
ALGEBRAIC[1] = 4.0*exp(-(STATES[0]+72.0)/18.0);
RATES[1] = ALGEBRAIC[0]*(1.0-STATES[1])-ALGEBRAIC[1]*STATES[1];
ALGEBRAIC[2] = 0.08*exp(-(STATES[0]+71.0)/19.0);
ALGEBRAIC[3] = 1.1/(exp(-(STATES[0]+44.0)/11.0)+1.0);
RATES[2] = ALGEBRAIC[2]*(1.0-STATES[2])-ALGEBRAIC[3]*STATES[2];
ALGEBRAIC[4] = 0.4/(1.0+exp(-(STATES[0]+28.0)/12.0));
ALGEBRAIC[5] = 0.13*exp(-(STATES[0]+70.0)/60.0);
RATES[3] = ALGEBRAIC[4]*(1.0-STATES[3])-ALGEBRAIC[5]*STATES[3];
ALGEBRAIC[6] = 0.11*exp(-(STATES[0]+60.0)/20.0);
ALGEBRAIC[7] = 0.9/(exp(-(STATES[0]+41.0)/13.0)+1.0);
RATES[4] = ALGEBRAIC[6]*(1.0-STATES[4])-ALGEBRAIC[7]*STATES[4];
ALGEBRAIC[8] = 0.13*exp((STATES[0]+62.0)/45.0);
ALGEBRAIC[9] = 0.7/(exp((STATES[0]+47.0)/14.0)+1.0);
RATES[5] = ALGEBRAIC[8]*(1.0-STATES[5])-ALGEBRAIC[9]*STATES[5];
ALGEBRAIC[10] = 0.05*exp(-(STATES[0]+58.0)/30.0);
ALGEBRAIC[11] = 0.3/(exp(-(STATES[0]+39.0)/15.0)+1.0);
RATES[6] = ALGEBRAIC[10]*(1.0-STATES[6])-ALGEBRAIC[11]*STATES[6];
ALGEBRAIC[12] = 0.02*exp((STATES[0]+66.0)/50.0);
ALGEBRAIC[13] = 0.1/(exp((STATES[0]+52.0)/16.0)+1.0);
RATES[7] = ALGEBRAIC[12]*(1.0-STATES[7])-ALGEBRAIC[13]*STATES[7];
ALGEBRAIC[14] = CONSTANTS[1]*pow(STATES[1], 3.0)*STATES[2]*(STATES[0]-45.0);
ALGEBRAIC[15] = CONSTANTS[2]*pow(STATES[3], 4.0)*(STATES[0]+85.0);
ALGEBRAIC[16] = CONSTANTS[3]*(STATES[0]+60.0-5.0*STATES[4]*STATES[5]*STATES[6]*STATES[7]);
RATES[0] = CONSTANTS[0]-ALGEBRAIC[14]-ALGEBRAIC[15]-ALGEBRAIC[16];
}
